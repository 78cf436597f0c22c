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


@pytest.mark.parametrize("name", ["cube", "cut_cube", "cut_sector"])
def test_shared_edges_take_mean_and_hall(oracle_mod, name):
    """E and the Hall EMF on every owned edge, those shared across a seam or an
    interface and those that also lie on the solid surface among them."""
    case = {"cube": lambda: cases.make_periodic_cube(n=(7, 6, 8), g=4, hall=True),
            "cut_cube": lambda: cases.make_split_cube(n=(9, 8, 10), split=(2, 2, 2), g=4, hall=True),
            "cut_sector": lambda: cases.make_split_sector(dims=(12, 9, 10), cuts=((5, 7), (4, 5), (10,)))}[name]()
    g = Mercury(case)
    o = oracle_mod.Oracle(case)
    try:
        g.prepare()
        o.prepare()
        np.testing.assert_array_equal(g.step(2), o.step(2))
        for field in ("E", "Ehall"):
            for a, axis in enumerate(("xi", "eta", "zeta")):
                for ib in range(case.nb):
                    m = case.blocks[ib].dims
                    own = (slice(None),) + tuple(slice(case.g, case.g + m[c] + (c != a)) for c in range(3))
                    n = f"{field}_{axis}"
                    np.testing.assert_array_equal(g.get(n, ib)[own], o.get(n, ib)[own], err_msg=f"{n}[{ib}]")
    finally:
        g.close()


def test_flux_shape_of_a_large_context_of_three_species():
    """Four cells per thread where their waves fill the chip four times over, whatever
    the number of species (3.2 M cells in the mixed form: 12 600 waves of 12 288)."""
    case = cases.make_shell(blocks=((160, 140, 144),), he=True)
    print(f"[case] {case.name} flux shape", flush=True)
    g = Mercury(case)
    try:
        assert g.flux_shape() == (0, 4)
        g.set_form(2)
        assert g.flux_shape() == (0, 4)
    finally:
        g.close()
