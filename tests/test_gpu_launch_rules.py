"""The launch shape and the streams a context chooses by its size."""
import numpy as np
import pytest

from mpcns_mercury_amd import cases
from mpcns_mercury_amd.hip import Mercury

pytestmark = pytest.mark.gpu


def test_flux_shape_follows_size_until_chosen():
    """Few cells: one per thread; a choice of the caller's outlives a change of form."""
    g = Mercury(cases.make_periodic_cube(n=(10, 8, 6), g=4))
    assert g.flux_shape() == (0, 1)
    g.set_form(2)
    assert g.flux_shape() == (0, 1)
    g.set_flux_shape(0, 3)
    g.set_form(1)
    assert g.flux_shape() == (0, 3)
    g.close()


@pytest.mark.parametrize("overlap", ["0", "1"])
@pytest.mark.parametrize("length", [1, 2, 4])
@pytest.mark.parametrize("integrator", [0, 1])
def test_streams_and_shapes_keep_every_bit(oracle_mod, monkeypatch, overlap, length, integrator):
    """One stream or two, and every length the rule can choose (over a block that
    none of them divides): three steps equal the oracle's."""
    monkeypatch.setenv("MERCURY_OVERLAP", overlap)
    case = cases.make_split_sector(dims=(13, 9, 10), cuts=((13,), (4, 5), (10,)))
    g = Mercury(case)
    o = oracle_mod.Oracle(case)
    try:
        g.prepare()
        o.prepare()
        g.set_flux_shape(0, length)
        np.testing.assert_array_equal(g.step(3, integrator), o.step(3, integrator))
        for name in ("U_H", "U_Na", "B_xi", "B_eta", "B_zeta", "J_cell", "PV_H", "RHS_H"):
            for ib in range(case.nb):
                np.testing.assert_array_equal(g.get(name, ib), o.get(name, ib), err_msg=f"{name}[{ib}]")
    finally:
        g.close()
