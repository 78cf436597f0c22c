"""The J reconstruction from its factors: the same bits as the stored weights, and
the stored weights whenever a caller may have changed them or the edge vectors."""
import numpy as np
import pytest

from mpcns_mercury_amd import cases
from mpcns_mercury_amd.hip import Mercury

pytestmark = pytest.mark.gpu


def _case():
    return cases.make_shell(blocks=((7, 6, 5), (5, 8, 6)))


def _jcell(g):
    g.op("jcell_t")
    return [g.get("J_cell", ib) for ib in range(g.case.nb)]


def test_factors_give_the_stored_weights_bits():
    g = Mercury(_case())
    g.prepare()
    g.step(2)
    a = _jcell(g)
    g.op("jcell")  # the per-function pass reads the 36 weights
    for ib in range(g.case.nb):
        np.testing.assert_array_equal(a[ib], g.get("J_cell", ib))
    g.close()


@pytest.mark.parametrize("field", ["Jcell_from_Jedge_w", "dr_xi", "dr_zeta"])
@pytest.mark.parametrize("how", ["upload", "graph", "address"])
def test_written_weights_are_used(field, how):
    """After a caller writes the weights (or an edge vector, which leaves the
    weights as they are), and after it has asked for the address of either, the
    stored weights are the ones that count, also in a step captured before."""
    g = Mercury(_case())
    g.prepare()
    if how == "graph":
        g.graph_capture(0)
    if how == "address":
        g.field_device(field, 1, 1)
    else:
        w = g.get(field, 1)
        w[1] *= 1.5
        g.set(field, 1, w)
    if how == "graph":
        g.graph_launch(1)
        a = [g.get("J_cell", ib) for ib in range(g.case.nb)]
        m, c = g.case.blocks[1].dims, g.case.g
        own = (slice(None), slice(c + 2, c + m[0]), slice(c, c + m[1]), slice(c, c + m[2]))  # the wall's sync zeroes two layers
    else:
        a, own = _jcell(g), Ellipsis
    g.op("jcell")
    np.testing.assert_array_equal(a[1][own], g.get("J_cell", 1)[own])
    g.close()
