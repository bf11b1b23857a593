"""The sweep's branches at the sizes where they can go wrong, against the
oracle: rows of even and odd number, columns entered again (a hole), a step
whose discriminant leaves the right half plane (items swept again), and lane
layouts with one, two, four and other numbers of lanes per column, with idle
lanes and padded energies.

FP64: every grid point within 1e-10 of the oracle relative to the field's
largest magnitude, the parity bar (a step rounds to 1e-15, and the sums of a
few hundred steps, energies and angles stay below 1e-13).  FP32 stepping: 1e-5,
a few hundred FP32 roundings (6e-8) of values of order one."""
import numpy as np
import pytest

from test_gpu_parity import rel

pytestmark = pytest.mark.gpu


def grain(ppxi, flux, geometry, temperature=0.4, angles=10, cutoff=8.0):
    return {
        "physics": {"temperature": temperature, "external_flux_quanta": flux,
                    "penetration_depth": -1.0, "gauge": "symmetric", "charge_sign": -1,
                    "crystal_axes_rotation": 0.1,
                    "order_parameter": {"dx2-y2": {"critical_temperature": 1.0},
                                        "s": {"critical_temperature": 0.4,
                                              "initial_phase_shift": 0.25}}},
        "geometry": geometry,
        "numerics": {"convergence_criterion": 1e-8, "energy_cutoff": cutoff, "norm": "l2",
                     "num_fermi_momenta": angles, "points_per_coherence_length": ppxi,
                     "vector_potential_error": 0.0},
        "accelerator": {"name": "picard", "step_size": 1.0}, "misc": {"seed": 3},
    }


def disc(radius, add=True, x=0.0, y=0.0):
    return {"disc": {"radius": radius, "center_x": x, "center_y": y, "add": add}}


def square(side):
    return {"regular_polygon": {"num_edges": 4, "side_length": side, "rotation": 0.06,
                                "center_x": 0.0, "center_y": 0.0, "add": True}}


# (name, config, lane layouts): 8 Ozaki energies at T = 0.4 and cutoff 8
CASES = {
    # the smallest grains: columns of a few rows, half of them shorter than
    # a pair of sites
    "tiny_disc": (grain(3.0, 0.5, [disc(1.2)]), [(1, 4, 16), (8, 2, 8)]),
    "odd_rows": (grain(5.0, 0.5, [disc(2.7)]), [(2, 4, 16), (3, 3, 16), (4, 2, 8), (7, 1, 4)]),
    "square": (grain(4.0, 1.0, [square(6.1)]), [(1, 4, 4), (2, 4, 8), (5, 2, 8), (16, 1, 4)]),
    # columns that leave the grain and enter it again, off centre
    "hole": (grain(6.0, 0.5, [square(6.0), disc(1.3, False, 0.4, -0.3)]),
             [(1, 4, 16), (2, 4, 16), (4, 3, 8), (8, 2, 8)]),
    # a Doppler shift of the order of the inverse lattice spacing: steps of
    # h |Re e| up to 3 take the root of a discriminant in the left half plane
    "strong_field": (grain(3.0, 60.0, [disc(3.0)]), [(1, 4, 16), (2, 4, 8), (8, 2, 8)]),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_sweep_paths_match_oracle(product, oracle, name):
    cfg, shapes = CASES[name]
    o = oracle.Oracle(cfg)
    o.initial_bulk()
    rng = np.random.default_rng(5)
    start = [d * (1 + 0.05 * rng.normal(size=d.shape)) * np.exp(0.3j * rng.normal(size=d.shape))
             for d in o.delta()]
    for c, d in enumerate(start):
        o.set_order_parameter(c, d)
    for _ in range(2):
        o.compute()
    want = (o.delta(True), o.current(), o.get("free_energy_per_area"))
    for shape in shapes:
        for precision, tol in (("fp64", 1e-10), ("mixed", 1e-5)):
            with product.Simulation(cfg) as s:
                s.set_sweep_shape(*shape, precision=precision)
                for c, d in enumerate(start):
                    s.set_order_parameter(c, d)
                for _ in range(2):
                    s.compute(precision)
                errs = (rel(s.order_parameter(1), want[0]), rel(s.current(), want[1]),
                        rel(s.results()["free_energy_per_area"], want[2]))
            print(name, shape, precision, ["%.1e" % e for e in errs])
            assert max(errs[:2]) < tol and errs[2] < 10 * tol
