"""Performance cases of the self-consistency path.

Each case is one call that a program makes on the framework in earnest: some
iterations of a solve with the fields read out afterwards (FP64 or mixed
precision, one grain or a batch), a Newton-Krylov step, a gradient of the
free energy, a Jacobian-vector product, iterations of the LDOS postprocess, a
vector-potential solve on host arrays.  Grain sizes, angles, temperatures and
cutoffs are those of the named workloads (superconga_amd/workloads.py), of the
reference's example configurations and of the tests, or lie between them.

The contexts are used as constructed, with the lane layout they come with.
"""
import math

import numpy as np
import torch

import superconga_amd as sa
from superconga_amd import workloads

# Floating-point operations a trajectory step cannot do without, each add,
# multiply, square root and reciprocal counted once: the midpoint step of the
# Riccati equation for one energy (10 for the discriminant, 24 for the complex
# square root, 24 for the quotient), and half of the Green-function sums of
# a site and energy (44), which both coherence functions share.
STEP_FLOPS = 80


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _grain(name, call, grain, size, ppxi, angles, temperature, cutoff, pairing, flux,
           penetration, accelerator, precision, iterations):
    return {"name": name, "call": call, "grain": grain, "size": size, "ppxi": ppxi,
            "angles": angles, "temperature": temperature, "cutoff": cutoff,
            "pairing": pairing, "flux": flux, "penetration": penetration,
            "accelerator": accelerator, "precision": precision, "iterations": iterations}


def listed():
    return [
        # the smallest solve of the named workloads: launches and the chain
        # of steps along one trajectory count, not throughput
        _grain("small_disc_fp64", "solve", "disc", 10.0, 10.0, 32, 0.5, 16.0, "s", 0.0, -1.0,
               "picard", "fp64", 4),
        _grain("small_disc_mixed", "solve", "disc", 10.0, 10.0, 32, 0.5, 16.0, "s", 0.0, -1.0,
               "picard", "mixed", 4),
        # an ordinary solve with a self-consistent vector potential
        _grain("vortex_disc_fp64", "solve", "disc", 12.5, 20.0, 64, 0.2, 16.0, "s", 2.0, 3.0,
               "congacc", "fp64", 8),
        # the flagship grain (1.3 million rotated sites, 128 angles, 28
        # energies), FP64 and with FP32 stepping
        _grain("octagon_fp64", "solve", "octagon", 25.0, 20.0, 128, 0.1, 32.0, "d", 0.0, 5.0,
               "anderson", "fp64", 8),
        _grain("octagon_mixed", "solve", "octagon", 25.0, 20.0, 128, 0.1, 32.0, "d", 0.0, 5.0,
               "anderson", "mixed", 8),
        # a parameter sweep's grains of uneven size iterated together
        {"name": "batch_fp64", "call": "batch", "count": 16, "sweep": 2024, "ppxi": 20.0,
         "precision": "fp64", "iterations": 4},
        # one Newton step with FP32 Jacobian-vector products, as a solve to a
        # tight residual takes several of
        _grain("newton_disc", "newton", "disc", 12.5, 10.0, 48, 0.3, 16.0, "d", 0.5, 4.0,
               "picard", "mixed", 1),
        # backward: free-energy gradient in the order parameter and the
        # vector potential; forward mode: an exact Jacobian-vector product
        _grain("gradient_square", "gradient", "square", 30.0, 20.0, 128, 0.3, 16.0, "d+is", 1.0,
               3.0, "anderson", "fp64", 1),
        _grain("jacobian_square", "jacobian", "square", 30.0, 20.0, 128, 0.3, 16.0, "d+is", 1.0,
               3.0, "anderson", "fp64", 1),
        # the LDOS postprocess: one block of 32 real energies, 720 angles
        _grain("ldos_disc", "ldos", "disc", 10.0, 15.0, 720, 0.3, 16.0, "d", 1.0, -1.0,
               "picard", "fp64", 2),
        # the vector-potential solve called on host arrays
        {"name": "poisson_506", "call": "poisson", "n": 506, "ppxi": 20.0},
    ]


def draw(rng):
    """One more case of the same ranges, no costlier than the octagon's."""
    call = rng.choice(["solve", "solve", "solve", "solve", "batch", "newton", "gradient",
                       "jacobian", "ldos", "poisson"])
    if call == "poisson":
        return {"call": call, "n": int(round(math.exp(rng.uniform(math.log(40), math.log(931))))),
                "ppxi": rng.choice([5.0, 8.0, 10.0, 15.0, 20.0])}
    if call == "batch":
        return {"call": call, "count": rng.randint(3, 14), "sweep": rng.randrange(1, 100000),
                "ppxi": rng.choice([8.0, 10.0, 15.0, 20.0]),
                "precision": rng.choice(["fp64", "fp64", "mixed"]),
                "iterations": rng.randint(1, 4)}
    while True:
        grain = rng.choice(["disc", "disc", "square", "octagon"])
        case = {
            "call": call, "grain": grain,
            "size": round(math.exp(rng.uniform(math.log(4.0), math.log(25.0)))
                          * (1.5 if grain == "square" else 1.0), 3),
            "ppxi": rng.choice([4.0, 5.0, 8.0, 10.0, 15.0, 20.0]),
            "angles": (rng.choice([180, 360, 720]) if call == "ldos" else
                       rng.choice([16, 24, 30, 32, 45, 48, 64, 96, 128])),
            "temperature": round(rng.uniform(0.1, 0.8), 3),
            "cutoff": rng.choice([8.0, 16.0, 16.0, 32.0]),
            "pairing": rng.choice(["s", "d", "d+is"]),
            "flux": rng.choice([0.0, 0.5, 1.0, 2.0]),
            "penetration": rng.choice([-1.0, 3.0, 5.0, 10.0]),
            "accelerator": rng.choice(["picard", "congacc", "anderson"]),
            "precision": "fp64", "iterations": 1}
        if call == "solve":
            case["precision"] = rng.choice(["fp64", "fp64", "mixed"])
            case["iterations"] = rng.choice([2, 4, 8])
        elif call == "newton":
            case["precision"] = "mixed"
        elif call == "ldos":
            case["iterations"] = 2
            case["penetration"] = -1.0
        if call in ("solve", "newton") and case["accelerator"] != "anderson" \
                and case["penetration"] > 0:
            case["accelerator"] = "congacc"
        if 5e6 < work(case)["flops"] < 2e12 and _n0(case) >= 30 \
                and case["angles"] * _n0(case) ** 2 * 2 < 2.2e8:
            return case


def tolerance(case):
    """Rounding alone.  FP64 sums taken in other lane layouts differ by up to
    1e-14 after eight iterations, and the accelerators amplify what a step of
    the recurrence rounds; FP32 stepping is 3e-5 off FP64 stepping in the
    current of an accelerated solve, and 4e-4 in a Newton step whose products
    are FP32 differences over 3e-4."""
    if case["call"] == "poisson":
        return {"rel": 1e-12}
    if case["call"] == "newton":
        return {"rel": 2e-3}
    if case["precision"] == "mixed":
        return {"rel": 1e-4}
    return {"rel": 1e-11}


def work(case):
    """Bytes: the state read and the results written once per iteration;
    flops: the trajectory steps of every angle and energy."""
    call = case["call"]
    if call == "poisson":
        n = case["n"]
        m = 1 << math.ceil(math.log2(2 * n - 1))
        return {"bytes": 4.0 * 8 * n * n, "flops": 2 * 5.0 * m * m * 2 * math.log2(m)}
    if call == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        for cfg in workloads.parameter_sweep(case["count"], case["sweep"], case["ppxi"]):
            g = cfg["geometry"][0]
            disc = g.get("disc")
            sub = {"call": "solve", "grain": "disc" if disc else "square",
                   "size": disc["radius"] if disc else g["regular_polygon"]["side_length"],
                   "ppxi": case["ppxi"], "angles": 64, "cutoff": 16.0, "pairing": "s",
                   "penetration": -1.0, "temperature": cfg["physics"]["temperature"],
                   "iterations": case["iterations"]}
            for k, x in work(sub).items():
                total[k] += x
        return total
    size, ppxi = case["size"], case["ppxi"]
    area = {"disc": math.pi * size * size, "square": size * size,
            "octagon": 2.0 * math.sqrt(2.0) * size * size}[case["grain"]]
    n0 = _n0(case)
    ne = 32 if call == "ldos" else _num_energies(case["temperature"], case["cutoff"])
    steps = 2.0 * ne * case["angles"] * area * ppxi * ppxi * case["iterations"]
    fields = 2 * (2 if case["pairing"] == "d+is" else 1) + (2 if case["penetration"] > 0 else 0)
    state = 2.0 * 8 * fields * n0 * n0 * case["iterations"]
    if call == "ldos":
        return {"bytes": state + 8.0 * 32 * n0 * n0 * case["iterations"], "flops": 70 * steps}
    # a reverse sweep takes the forward steps and twice as much for their
    # adjoints, a tangent sweep as much again as the forward steps; a Newton
    # step evaluates the map at least twice per Krylov direction
    factor = {"solve": 1.0, "gradient": 3.0, "jacobian": 2.0, "newton": 6.0}[call]
    return {"bytes": state * factor, "flops": STEP_FLOPS * steps * factor}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _extent(case):
    """The grain's larger side in coherence lengths."""
    size = case["size"]
    return {"disc": 2.0 * size, "square": size,
            "octagon": 2.0 * size * math.cos(math.pi / 8)}[case["grain"]]


def _n0(case):
    """Sites a side of the reference grid (rounding can add one to a polygon's)."""
    return math.ceil(_extent(case) * case["ppxi"]) + 6


def _largest_pole(n):
    """The largest of n Ozaki poles: the inverse of the smallest positive
    eigenvalue of a symmetric tridiagonal matrix of order 2 n."""
    i = np.arange(2 * n - 1)
    e = 0.5 / np.sqrt((2.0 * i + 1.0) * (2.0 * i + 3.0))
    w = np.linalg.eigvalsh(np.diag(e, 1) + np.diag(e, -1))
    return 1.0 / w[w > 0].min()


def _num_energies(temperature, cutoff):
    target = 2.0 * math.pi * cutoff / temperature
    n = 1
    while _largest_pole(n) <= target:
        n += 1
    return n


def _config(case):
    size = case["size"]
    if case["grain"] == "disc":
        geometry = {"disc": {"radius": size, "center_x": 0.0, "center_y": 0.0, "add": True}}
    else:
        n = 4 if case["grain"] == "square" else 8
        side = size if n == 4 else 2.0 * size * math.sin(math.pi / 8)
        geometry = {"regular_polygon": {"num_edges": n, "side_length": side, "rotation": 0.0,
                                        "center_x": 0.0, "center_y": 0.0, "add": True}}
    op = {"s": {"s": {"critical_temperature": 1.0}},
          "d": {"dx2-y2": {"critical_temperature": 1.0}},
          "d+is": {"dx2-y2": {"critical_temperature": 1.0},
                   "s": {"critical_temperature": 0.5}}}[case["pairing"]]
    accelerator = {"picard": {"name": "picard", "step_size": 1.0},
                   "congacc": {"name": "congacc"},
                   "anderson": {"name": "anderson", "rank": 8, "step_size": 1.0}}
    return {
        "physics": {"temperature": case["temperature"], "external_flux_quanta": case["flux"],
                    "penetration_depth": case["penetration"], "gauge": "symmetric",
                    "charge_sign": -1, "crystal_axes_rotation": 0.125,
                    "order_parameter": op},
        "geometry": [geometry],
        "numerics": {"convergence_criterion": 1e-14, "energy_cutoff": case["cutoff"],
                     "norm": "l2", "num_fermi_momenta": case["angles"],
                     "points_per_coherence_length": case["ppxi"], "vector_potential_error": 0.0,
                     "num_iterations_burnin": 0, "num_iterations_min": 0,
                     "num_iterations_max": 10000},
        "accelerator": accelerator[case["accelerator"]], "misc": {"seed": 1},
    }


def _waves(rng, n, amplitude, count=6):
    """A smooth random field on the n x n grid: a few long waves."""
    x = np.linspace(-1.0, 1.0, n)
    out = np.zeros((n, n))
    for _ in range(count):
        kx, ky = rng.uniform(-3.0, 3.0, 2)
        out += rng.normal() * np.cos(kx * x[None, :] + ky * x[:, None] + rng.uniform(0, 6.28))
    return amplitude * out / math.sqrt(count)


def _order_parameter(case, n, seed):
    """Order parameters (components, N0, N0) as a solve meets them: the bulk
    amplitude with slow variations of size and phase and 1% noise."""
    rng = np.random.default_rng([int(seed), 7])
    bulk = 0.2807 * math.sqrt(1.0 - case["temperature"] ** 3)
    comps = [0.86 * bulk, 0.2j * bulk] if case["pairing"] == "d+is" else [
        bulk if case["pairing"] == "s" else 0.86 * bulk]
    phase = _waves(rng, n, 0.4)
    out = []
    for b in comps:
        noise = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
        out.append(b * (1.0 + _waves(rng, n, 0.1) + 0.01 * noise) * np.exp(1j * phase))
    return np.stack(out)


def _vector_potential(n, seed):
    rng = np.random.default_rng([int(seed), 8])
    return np.stack([_waves(rng, n, 0.01), _waves(rng, n, 0.01)])


def prepare(case, seed):
    call = case["call"]
    if call == "poisson":
        rng = np.random.default_rng([int(seed), 9])
        n = case["n"]
        y, x = np.mgrid[0:n, 0:n] - 0.5 * (n - 1)
        inside = x * x + y * y <= (0.5 * n - 3) ** 2
        j = np.stack([(_waves(rng, n, 0.1) + 0.001 * rng.normal(size=(n, n))) * inside
                      for _ in range(2)])
        return {"call": call, "j": j, "h": 1.0 / case["ppxi"], "sites": int(inside.sum())}
    if call == "batch":
        configs = workloads.parameter_sweep(case["count"], case["sweep"], case["ppxi"])
        for c in configs:
            c["misc"]["seed"] = int(seed)
        batch = sa.Batch(configs)
        return {"call": call, "batch": batch, "precision": case["precision"],
                "iterations": case["iterations"]}
    cfg = _config(case)
    if call == "ldos":
        post = workloads.postprocess_config(case["angles"], 32, 32)
        post["numerics"]["convergence_criterion"] = 1e-14
        sim = sa.Spectroscopy(cfg, post)
    else:
        sim = sa.Simulation(cfg)
    state = {"call": call, "sim": sim, "precision": case["precision"],
             "iterations": case["iterations"], "field": case["penetration"] > 0,
             "delta": _order_parameter(case, sim.N0, seed), "a": _vector_potential(sim.N0, seed)}
    for c, d in enumerate(state["delta"]):
        sim.set_order_parameter(c, d)
    if state["field"]:
        sim.set_vector_potential(*state["a"])
    if call == "jacobian":
        state["v"] = _order_parameter(case, sim.N0, int(seed) + 1000)
        state["va"] = _vector_potential(sim.N0, int(seed) + 1000)
    if call in ("gradient", "jacobian", "newton"):
        # the boundary values such a call finds: those of an iteration
        sim.burnin("fp64")
        state["boundary"] = [sim.boundary(0, d) for d in (0, 1)]
    if call == "newton":
        # all Krylov directions of one cycle
        sim.set_newton_options(restarts=1, eta_max=1e-4)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    call = state["call"]
    if call == "poisson":
        return sa.poisson_solve(state["j"], state["h"], state["sites"])
    n = state.get("iterations")
    if call == "batch":
        batch = state["batch"]
        batch.run(burnin=0, nmin=n, nmax=n, precision=state["precision"])
        grains = [batch.grain(i) for i in range(len(batch))]
        return {"delta": [g.order_parameter(1) for g in grains],
                "free_energy": np.array([g.results()["free_energy_per_area"] for g in grains])}
    sim = state["sim"]
    if call == "solve":
        # n further iterations of the solve, then its fields
        sim.run(burnin=0, nmin=n, nmax=n, precision=state["precision"])
        out = {"delta": sim.order_parameter(1), "current": sim.current(),
               "free_energy": sim.results()["free_energy_per_area"]}
        if state["field"]:
            out["a"] = sim.vector_potential(1)
        return out
    if call == "ldos":
        sim.run(burnin=0, nmin=n, nmax=n, precision=state["precision"])
        return sim.ldos()
    if call == "jacobian":
        return sim.jacobian_vector(state["v"], state["va"] if state["field"] else None)
    # a new order parameter (and vector potential) on a grain that is kept
    for c, d in enumerate(state["delta"]):
        sim.set_order_parameter(c, d)
    if state["field"]:
        sim.set_vector_potential(*state["a"])
    if call == "gradient":
        return sim.free_energy_gradient(vector_potential=state["field"])
    for d in (0, 1):
        sim.set_boundary(d, state["boundary"][d])
    report = sim.newton_krylov(max_newton=1, krylov_dim=8, tol=1e-12,
                               jvp_precision=state["precision"])
    return {"delta": sim.order_parameter(0), "residual": report["residual"],
            "a": sim.vector_potential(0) if state["field"] else None}


# ---------------------------------------------------------------------------
# the same in 64 bits with plain torch and numpy
# ---------------------------------------------------------------------------
def exact(case, seed):
    """The solves of discs by plain iteration without an induced vector
    potential, and the vector-potential solve.  The others have none: an
    accelerated solve, an adjoint or a Newton step restated here would be a
    second framework, and the large grains take minutes."""
    if case["call"] == "poisson":
        return _exact_poisson(prepare(case, seed))
    if case["call"] == "solve" and case["grain"] == "disc" and case["penetration"] <= 0 \
            and case["accelerator"] == "picard" and case["angles"] * _n0(case) < 40000:
        return _exact_disc(case, seed)
    return None


def _exact_poisson(state):
    j, h = state["j"], state["h"]
    n = j.shape[-1]
    # the lattice kernel: analytic cell integrals of the logarithm,
    # symmetrised, its mean moved into the constant part
    i = np.arange(n, dtype=np.float64)

    def alpha(a, b):
        return a * b * (2.0 * np.log(np.hypot(a, b)) - math.log(2.0))

    def beta(a, b):
        return 0.5 * ((2.0 - a + b) * (a + b) - 2.0) * np.arctan(a / b)

    q = np.zeros((n, n))
    for sj in (-1, 1):
        for si in (-1, 1):
            a, b = 1.0 + 2.0 * si * i[None, :], 1.0 + 2.0 * sj * i[:, None]
            q += 0.25 * (alpha(a, b) + beta(a, b) + beta(b, a))
    g = 0.5 * (q + q.T) / (4.0 * math.pi)
    g += (2.0 * math.log(h) - math.log(2.0) - 3.0) / (4.0 * math.pi)
    m = 2 * n
    full = np.zeros((m, m))
    full[:n, :n] = g
    full[n + 1:, :n] = g[1:][::-1]
    full[:, n + 1:] = full[:, 1:n][:, ::-1]
    spectrum = np.fft.rfft2(full)
    out = np.empty_like(j)
    for d in range(2):
        src = np.zeros((m, m))
        src[:n, :n] = j[d] - j[d].sum() / state["sites"]
        out[d] = -h * h * np.fft.irfft2(np.fft.rfft2(src) * spectrum, s=(m, m))[:n, :n]
    return out


def _exact_disc(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f8, c16 = torch.float64, torch.complex128
    na, T, ppxi = case["angles"], case["temperature"], case["ppxi"]
    h, n0 = 1.0 / ppxi, _n0(case)
    n1 = n0 + 2 * math.ceil(0.5 * (math.sqrt(2.0) - 1.0) * n0)
    radius = 0.5 * (_extent(case) * ppxi / n0) * (n0 - 1)
    # Ozaki poles and residues
    ne = _num_energies(T, case["cutoff"])
    i = np.arange(2 * ne - 1)
    e = 0.5 / np.sqrt((2.0 * i + 1.0) * (2.0 * i + 3.0))
    w, z = np.linalg.eigh(np.diag(e, 1) + np.diag(e, -1))
    pole = 1.0 / w[w > 0]
    res = (0.5 * z[0, w > 0] * pole) ** 2
    energy = pole * T / (2.0 * math.pi)
    sum_inverse = T * float(np.sum(res / energy))
    # Fermi surface
    k = np.arange(na)
    polar = math.pi * 2.0 * k / na + 0.5 * math.pi
    polar = np.where(polar >= 2.0 * math.pi, polar - 2.0 * math.pi, polar)
    theta = polar - 0.5 * math.pi
    if na % 4 == 0:
        weight = np.where(k % 4 == 0, 28.0, np.where(k % 2 == 0, 24.0, 64.0)) / 45.0
    elif na % 3 == 0:
        weight = np.where(k % 3 == 0, 6.0, 9.0) / 8.0
    elif na % 2 == 0:
        weight = np.where(k % 2 == 0, 2.0, 4.0) / 3.0
    else:
        weight = np.ones(na)
    weight = weight / na
    vx, vy = np.cos(polar), np.sin(polar)

    def trig(angle):  # cosines and sines of single-precision angles
        a = [float(np.float32(t)) for t in angle]
        return (np.array([float(np.float32(math.cos(t))) for t in a]),
                np.array([float(np.float32(math.sin(t))) for t in a]))

    op_trig = trig(-theta[(-k) % na].astype(np.float32))
    back_trig = trig(-theta.astype(np.float32))
    basis, coupling, tcs = [], [], []
    for c in range(2 if case["pairing"] == "d+is" else 1):
        d_wave = case["pairing"] != "s" and c == 0
        r = 2.0 * math.pi * 0.125
        rx, ry = vx * math.cos(r) - vy * math.sin(r), vx * math.sin(r) + vy * math.cos(r)
        norm = 1.0 / math.sqrt(np.sum((vx * vx - vy * vy) ** 2 * weight)) if d_wave else \
            1.0 / math.sqrt(np.sum(weight))
        basis.append((rx * rx - ry * ry if d_wave else np.ones(na)) * norm)
        tc = 0.5 if c == 1 else 1.0
        tcs.append(tc)
        coupling.append(0.5 * T / (math.log(T / tc) + sum_inverse))

    def labels(n):  # 1 inside, 2 lowest, 3 highest site of a column
        x = np.arange(-1, n + 1) - 0.5 * (n - 1)
        inside = (x[None, :] ** 2 + x[:, None] ** 2 <= radius * radius).astype(int)
        row = inside[:, :-2] + inside[:, 1:-1] + inside[:, 2:] > 1
        low, mid, high = row[:-2], row[1:-1], row[2:]
        return np.where(mid & low & high, 1, np.where(mid & high & ~low, 2,
                                                      np.where(mid & low & ~high, 3, 0)))

    # a centred disc has the same labels in every rotated frame
    lab1 = labels(n1)
    domain = torch.tensor(labels(n0) > 0, device=dev)
    cols = np.where((lab1 == 2).any(0))[0]
    low, high = (lab1[:, cols] == 2).argmax(0), (lab1[:, cols] == 3).argmax(0)
    off = 0.5 * (n1 - 1)
    xc = cols - off

    def crossing(row):
        y = row - off
        d = np.sqrt(radius * radius - xc * xc) - np.abs(y)
        return np.abs(d), -xc / radius, np.where(y <= 0, -(y - d), -(y + d)) / radius

    def rot(a, x, y):
        return x * np.cos(a) - y * np.sin(a), x * np.sin(a) + y * np.cos(a)

    def stencil(gamma):
        """Sources (angle, column) and weights of every entry's value."""
        row = low if gamma else high
        dist, nx, ny = crossing(row)
        mx, my = rot(-theta[:, None], vx[:, None], vy[:, None])
        two = 2.0 * (mx * nx + my * ny)

        def at(rx, ry):
            gx, gy = rot(theta[:, None], rx, ry)
            phi = np.mod(np.arctan2(gy, gx) - 0.5 * math.pi, 2.0 * math.pi)
            f = na * phi / (2.0 * math.pi)
            py = row - (1 if gamma else -1) * dist - off
            ks, xs, ws = [], [], []
            for r in (0, 1):
                kk = (f.astype(int) + r) % na
                wk = f - np.floor(f) if r else 1.0 - (f - np.floor(f))
                qx, _ = rot(theta[:, None] - theta[kk], xc[None, :], py[None, :])
                qx = qx + off
                for t in (0, 1):
                    xx = qx.astype(int) + t
                    wx = qx - np.floor(qx) if t else 1.0 - (qx - np.floor(qx))
                    ok = (xx >= 0) & (xx < n1) & np.isin(xx, cols)
                    ks.append(kk)
                    xs.append(np.clip(xx, 0, n1 - 1))
                    ws.append(np.where(ok, wk * wx, 0.0))
            return np.stack(ks), np.stack(xs), np.stack(ws)

        a, b = at(mx - two * nx, my - two * ny), at(-mx + 0.0 * nx, -my + 0.0 * ny)
        none = a[2].sum(0) < 1e-7
        ks, xs, ws = (np.where(none, q, p) for p, q in zip(a, b))
        total = ws.sum(0)
        ws = np.where(total > 0, ws / np.where(total > 0, total, 1.0), 0.0)
        return (torch.tensor(ks, device=dev), torch.tensor(xs, device=dev),
                torch.tensor(ws, device=dev))

    stencils = {True: stencil(True), False: stencil(False)}

    def boundary(out, gamma):  # in-values from out-values (na, n1, ne)
        ks, xs, ws = stencils[gamma]
        return (out[ks, xs] * ws[..., None]).sum(0)

    def cell(m, n, c, s):
        """Cells and fractions of the sites of an m grid in an n grid."""
        x = torch.arange(m, device=dev, dtype=f8) + (n - m) / 2.0 - (n - 1) / 2.0
        c, s = (torch.tensor(v, device=dev).reshape(-1, 1, 1) for v in (c, s))
        X = (x[None, None, :] * c - x[None, :, None] * s) + (n - 1) / 2.0
        Y = (x[None, None, :] * s + x[None, :, None] * c) + (n - 1) / 2.0
        xi, yi = X.trunc().long(), Y.trunc().long()
        ok = (xi >= 0) & (xi + 1 < n) & (yi >= 0) & (yi + 1 < n)
        return xi.clamp(0, n - 2), yi.clamp(0, n - 2), X - xi, Y - yi, ok

    def sample(grid, where, frame=None):
        xi, yi, fx, fy, ok = where
        if frame is None:
            at = lambda y, x: grid[y, x]  # noqa: E731
        else:
            at = lambda y, x: grid[frame, y, x]  # noqa: E731
        a = (1.0 - fx) * at(yi, xi) + fx * at(yi, xi + 1)
        b = (1.0 - fx) * at(yi + 1, xi) + fx * at(yi + 1, xi + 1)
        return torch.where(ok, (1.0 - fy) * a + fy * b, torch.zeros((), dtype=a.dtype, device=dev))

    def extend(grid, inside):
        """Outside sites take the mean of their nearest inside ones (5 x 5)."""
        out = torch.where(inside, grid, torch.zeros((), dtype=grid.dtype, device=dev))
        pad = torch.nn.functional.pad
        value, mask = pad(out, (2, 2, 2, 2)), pad(inside, (2, 2, 2, 2))
        n, done = grid.shape[-1], inside.clone()
        for d2 in (1, 2, 4, 5, 8):
            total, count = torch.zeros_like(out), torch.zeros(inside.shape, device=dev, dtype=f8)
            for dy in range(-2, 3):
                for dx in range(-2, 3):
                    if dx * dx + dy * dy == d2:
                        total += value[..., 2 + dy:2 + dy + n, 2 + dx:2 + dx + n]
                        count += mask[..., 2 + dy:2 + dy + n, 2 + dx:2 + dx + n]
            new = ~done & (count > 0)
            out = torch.where(new, total / count.clamp(min=1.0), out)
            done |= new
        return out

    inside1 = torch.tensor(lab1 > 0, device=dev)
    num_grain = int(domain.sum())
    field = -0.5 * math.pi * case["flux"] / (h * h * num_grain)  # charge -1, symmetric gauge
    xs = (torch.arange(n1, device=dev, dtype=f8) - off) * h
    t8 = lambda v: torch.tensor(v, device=dev, dtype=f8)  # noqa: E731
    ct, st = t8(np.cos(theta)).reshape(-1, 1, 1), t8(np.sin(theta)).reshape(-1, 1, 1)
    px, py = xs[None, None, :] * ct - xs[None, :, None] * st, \
        xs[None, None, :] * st + xs[None, :, None] * ct
    shift = field * (t8(vx).reshape(-1, 1, 1) * -py + t8(vy).reshape(-1, 1, 1) * px)
    into = cell(n1, n0, *op_trig)
    omega, residue = t8(energy), t8(res)
    delta = torch.where(domain, torch.tensor(_order_parameter(case, n0, seed), device=dev), 0.0)

    def rotated(d):
        return sum(t8(b).reshape(-1, 1, 1) * sample(extend(x, domain), into)
                   for b, x in zip(basis, d))

    def step(d, es, y0, hh):
        """Implicit midpoint step from y0 over hh (broadcast)."""
        s = 1j * hh
        a = s * d.conj() / 4.0
        se = s * (es + 1j * omega)
        b = 2.0 * a * y0 + se - 1.0
        c = (a * y0 + se + 1.0) * y0 + s * d
        return 2.0 * c / (torch.sqrt(b * b - 4.0 * a * c) - b)

    ci = torch.tensor(cols, device=dev)
    rows = {True: torch.tensor(low, device=dev), False: torch.tensor(high, device=dev)}
    dists = {g: t8(crossing(r)[0])[None, :, None] for g, r in ((True, low), (False, high))}
    bin_, first = None, True
    for it in range(case["iterations"]):
        D = rotated(delta)
        if first:  # bulk solutions leave the grain, and the boundary turns them
            first, out = False, {}
            for gamma in (True, False):
                r = rows[not gamma]
                d, es = D[:, r, ci][..., None], shift[:, r, ci][..., None]
                ep = es + 1j * omega
                den = ep + 1j * torch.sqrt(d.abs() ** 2 - ep * ep)
                out[gamma] = torch.zeros((na, n1, ne), dtype=c16, device=dev)
                out[gamma][:, ci] = (-d if gamma else d.conj()) / den
            bin_ = {g: boundary(out[g], g) for g in (True, False)}
        store = torch.zeros((na, n1, len(cols), ne), dtype=c16, device=dev)
        green = torch.zeros((na, n1, n1, 4), dtype=f8, device=dev)
        new_out = {}
        for gamma in (False, True):
            sign = 1 if gamma else -1
            begin, end = rows[gamma], rows[not gamma]
            dd = D[:, :, ci] if gamma else -D[:, :, ci].conj()
            ss = shift[:, :, ci]
            y = torch.zeros((na, len(cols), ne), dtype=c16, device=dev)
            out = torch.zeros((na, n1, ne), dtype=c16, device=dev)
            order = range(int(low.min()), int(high.max()) + 1)
            for t in (order if gamma else reversed(order)):
                d, es = dd[:, t][..., None], ss[:, t][..., None]
                dm = 0.5 * (d + dd[:, t - sign][..., None])
                em = 0.5 * (es + ss[:, t - sign][..., None])
                stepped = step(dm, em, y, h)
                entered = step(d, es, bin_[gamma], dists[gamma] * h)
                live = ((t - begin) * sign >= 0) & ((end - t) * sign >= 0)
                y = torch.where((begin == t)[None, :, None], entered, stepped)
                y = torch.where(live[None, :, None], y, torch.zeros((), dtype=c16, device=dev))
                left = step(d, es, y, dists[not gamma] * h)
                out[:, ci] = torch.where((end == t)[None, :, None], left, out[:, ci])
                if not gamma:
                    store[:, t] = y
                    continue
                gt = store[:, t]
                p = y * gt
                F = 2j / (1.0 + p)
                u, v = gt - y, y + gt
                sums = torch.stack([(residue * (F * u).real).sum(-1),
                                    -(residue * (F * v).imag).sum(-1),
                                    -(residue * F.real).sum(-1),
                                    d[..., 0].real * (residue * u.imag).sum(-1)
                                    + d[..., 0].imag * (residue * v.real).sum(-1)], -1)
                green[:, t, ci] = torch.where(live[None, :, None], sums, 0.0)
            new_out[gamma] = out
        total = torch.zeros((2 * len(basis) + 3, n0, n0), dtype=f8, device=dev)
        for kk in range(na):
            back = cell(n0, n1, back_trig[0][kk:kk + 1], back_trig[1][kk:kk + 1])
            g = [sample(extend(green[kk, :, :, q], inside1), [b[0] for b in back])
                 for q in range(4)]
            for c, b in enumerate(basis):
                total[2 * c] += g[0] * (b[kk] * weight[kk])
                total[2 * c + 1] += g[1] * (b[kk] * weight[kk])
            total[-3] += g[2] * (vx[kk] * weight[kk])
            total[-2] += g[2] * (vy[kk] * weight[kk])
            total[-1] += g[3] * weight[kk]
        total = torch.where(domain, total, 0.0)
        free = T * float(total[-1].sum())
        for c, tc in enumerate(tcs):
            free += float((delta[c].abs() ** 2).sum()) * (math.log(T / tc) + sum_inverse)
        current = total[-3:-1] * (-2.0 * T)
        delta = torch.stack([coupling[c] * torch.complex(total[2 * c], total[2 * c + 1])
                             for c in range(len(basis))])
        bin_ = {g: boundary(new_out[g], g) for g in (True, False)}
    return {"delta": delta, "current": current, "free_energy": free / num_grain}
