"""The J reconstruction from its factors: the same bits as the stored weights, and
the stored weights whenever a caller may have changed them or the edge vectors."""
import numpy as np
import pytest

from mpcns_mercury_amd import cases
from mpcns_mercury_amd.hip import Mercury

import hipmem
import restart_format as rf

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
    weights as they are), by an upload or at the address it has asked for, the
    stored weights are the ones that count, also in a step captured before."""
    g = Mercury(_case())
    g.prepare()
    g.step(2)  # J starts at zero
    if how == "graph":
        g.graph_capture(0)
    before = _jcell(g)[1]
    w = g.get(field, 1)
    w[1] *= 1.5
    if how == "address":
        hipmem.copy_in(g.field_device(field, 1, 1), w[1])
    else:
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
    if how != "graph":
        assert (a[1] != before).any() == (field == "Jcell_from_Jedge_w")
    g.close()


@pytest.mark.parametrize("field", ["Jcell_from_Jedge_w", "dr_eta"])
def test_weights_of_a_restart_file_are_used(tmp_path, field):
    """A restart file may hold any field of the catalogue; weights or edge vectors
    that it brings are the caller's, as uploaded ones are."""
    g = Mercury(_case())
    g.prepare()
    g.step(2)  # J starts at zero
    loc = rf.LOC_CODE["cell" if field[0] == "J" else "ey"]
    blocks = []
    for ib in range(g.case.nb):
        hi = [m + 1 - d + g.case.g for m, d in zip(g.case.blocks[ib].dims, rf.DELTA_OF_CODE[loc])]
        w = g.get(field, ib)[(slice(None),) + tuple(slice(0, h + g.case.g) for h in hi)]
        blocks.append(((-g.case.g,) * 3, hi, 1.25 * w))
    p = tmp_path / "weights.bin"
    rf.write_restart(p, 0, 0.0, g.case.nb, [(field, loc, blocks[0][2].shape[0], g.case.g, blocks)])
    before = _jcell(g)
    g.read_restart(p)
    a = _jcell(g)
    g.op("jcell")
    for ib in range(g.case.nb):
        np.testing.assert_array_equal(a[ib], g.get("J_cell", ib))
    if field[0] == "J":
        assert any((x != y).any() for x, y in zip(a, before))
    g.close()
