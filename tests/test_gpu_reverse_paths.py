"""The reverse sweep of the free energy and the transpose of the site fields at
the sizes where their kernels can go wrong, against the oracle's adjoint: grids
below, at and above a tile of 16 x 16 sites, columns of every length about a
segment of four sites (a disc and a grain whose columns are entered again), and
energies that fill a lane's four or leave some over.

Every grid point within 1e-10 of the largest entry, the bar of
test_gpu_gradient.py (a step and its adjoint round to 1e-15, and the sums of a
few hundred steps, energies and angles stay below 1e-13)."""
import numpy as np
import pytest

import cases
from test_gpu_gradient import TOL, fresh_pair, state

pytestmark = pytest.mark.gpu


def grain(sites, temperature, hole=False):
    """A disc (with a hole off its centre) on a grid of `sites` sites a side."""
    components = [{"disc": {"radius": 0.5, "center_x": 0.0, "center_y": 0.0, "add": True}}]
    if hole:
        components.append({"disc": {"radius": 0.14, "center_x": 0.08, "center_y": -0.05,
                                    "add": False}})
    return cases.base(temperature=temperature, flux=0.7, lam=3.0, angles=10, ppxi=2.0,
                      width=(sites - 6) / 2.0,
                      order_parameter={"dx2-y2": {"critical_temperature": 1.0}},
                      components=components)


@pytest.mark.parametrize("sites,temperature,hole", [
    (15, 0.5, False), (16, 0.3, False), (17, 0.8, False), (32, 0.5, True), (33, 0.3, True),
    (49, 0.2, False)])
def test_reverse_sweep_matches_oracle(product, oracle, sites, temperature, hole):
    cfg = grain(sites, temperature, hole)
    d, a = state(product, cfg, 1)
    s, o = fresh_pair(product, oracle, cfg, d, a)
    print("sites a side", s.N0)
    assert abs(s.N0 - sites) <= 1
    f, g, ga = s.free_energy_gradient(vector_potential=True)
    fo, go, gao = o.free_energy_gradient(vector_potential=True)
    err = np.max(np.abs(g - go)) / np.max(np.abs(go))
    err_a = np.max(np.abs(ga - gao)) / np.max(np.abs(gao))
    print("gradient error %.1e of max, in A %.1e" % (err, err_a))
    assert abs(f - fo) <= 1e-12 * abs(fo)
    assert err < TOL and err_a < TOL
    s.close()
