"""Every sync group on random values in every box point, against the oracle's
phase by phase sync, bit for bit.

The device writes each changed value from where it comes from among the values
before the sync, in one launch per sync; the oracle runs the handlers, the corner
defaults, the halo stages and the owner copies one after another.  Random values
everywhere tell a value taken one phase too early or too late, which equal
copies of shared values would hide."""
import numpy as np
import pytest

from mpcns_mercury_amd import cases
from mpcns_mercury_amd.hip import Mercury, field_info

pytestmark = pytest.mark.gpu

TOPOLOGIES = {
    "cube": lambda: cases.make_periodic_cube(n=(7, 9, 6), g=4),
    "cube_smallest": lambda: cases.make_periodic_cube(n=(4, 4, 4), g=4),  # every ghost layer is a whole period
    "cut_cube": lambda: cases.make_split_cube(n=(9, 8, 10), split=(2, 2, 2), g=4),
    "shell": lambda: cases.make_shell(scale=0.1),
    "thin_shell": lambda: cases.make_shell(blocks=((3, 4, 5), (4, 3, 3))),
    "he_shell": lambda: cases.make_shell(scale=0.1, he=True),
    "cut_sector": lambda: cases.make_split_sector(dims=(12, 9, 10), cuts=((5, 7), (4, 5), (10,))),
    "cubed_sphere_rule0": lambda: cases.make_cubed_sphere(6, 5, rule=0),
    "cubed_sphere_rule1": lambda: cases.make_cubed_sphere(6, 5, rule=1),
}
EDGE = lambda n: [f"{n}_xi", f"{n}_eta", f"{n}_zeta"]  # noqa: E731
GROUPS = {"sync_ucell": ["U_H", "U_Na"], "sync_bface": EDGE("B"), "sync_badd": EDGE("Badd"), "sync_eedge": EDGE("E"),
          "sync_ehall": EDGE("Ehall"), "sync_jedge": EDGE("J"), "sync_bcell": ["B_cell", "Bind_cell"], "sync_jcell": ["J_cell"]}


@pytest.mark.parametrize("topology", list(TOPOLOGIES))
def test_sync_of_random_values(oracle_mod, topology):
    case = TOPOLOGIES[topology]()
    print(f"[case] {case.name} dims={[b.dims for b in case.blocks]}", flush=True)
    rng = np.random.default_rng(5)
    g = Mercury(case)
    o = oracle_mod.Oracle(case)
    try:
        for op, names in GROUPS.items():
            if op == "sync_ucell" and case.phys.n_species >= 3:
                names = names + ["U_He"]
            for name in names:
                for ib in range(case.nb):
                    v = rng.uniform(0.1, 2.0, (field_info(name)[1],) + case.box(ib))
                    g.set(name, ib, v)
                    o.set(name, ib, v)
            g.op(op)
            o.op(op, 0)
            for name in names:
                for ib in range(case.nb):
                    np.testing.assert_array_equal(g.get(name, ib), o.get(name, ib), err_msg=f"{op} {name}[{ib}]")
    finally:
        g.close()


def test_ensemble_syncs_like_its_runs():
    """An ensemble's far-field states are per run: each block's sync equals the
    same sync in the run's own context."""
    runs = [cases.make_ensemble_run(r, scale=0.12) for r in range(3)]
    e = Mercury(cases.concat_runs(runs))
    rng = np.random.default_rng(6)
    base = 0
    data = {}
    for op, names in GROUPS.items():
        for name in names:
            for ib in range(sum(c.nb for c in runs)):
                data[name, ib] = rng.uniform(0.1, 2.0, (field_info(name)[1],) + e.case.box(ib))
                e.set(name, ib, data[name, ib])
        e.op(op)
    for c in runs:
        m = Mercury(c)
        for op, names in GROUPS.items():
            for name in names:
                for ib in range(c.nb):
                    m.set(name, ib, data[name, base + ib])
            m.op(op)
            for name in names:
                for ib in range(c.nb):
                    np.testing.assert_array_equal(e.get(name, base + ib), m.get(name, ib), err_msg=f"{op} {name}[{ib}]")
        base += c.nb
        m.close()
    e.close()


def _walled(faces, blocks=((7, 6, 5), (5, 8, 6)), he=False):
    """The shell's sectors with solid surfaces on the listed faces of each block."""
    case = cases.make_shell(blocks=blocks, he=he)
    for b, on in zip(case.blocks, faces):
        b.bc = tuple(cases.BC_WALL if f in on else cases.BC_FARFIELD for f in range(6))
    return case


def _thin(case, n):
    """Block 0 cut to its first n cells along the first axis."""
    b, end = case.blocks[0], n + 1 + 2 * case.g
    b.dims, b.nodes = (n,) + tuple(b.dims[1:]), np.ascontiguousarray(b.nodes[:, :n + 1])
    case.fields[0] = {k: np.ascontiguousarray(v[:, :end]) for k, v in case.fields[0].items()}
    return case


WALLS = {
    "adjacent": lambda he: _walled([(0, 2), (0,)], he=he),
    "adjacent_upper": lambda he: _walled([(3, 5), (1,)], he=he),
    "three": lambda he: _walled([(0, 3, 4), ()], he=he),
    "six": lambda he: _walled([range(6), (2, 4)], he=he),
    "opposite": lambda he: _walled([(0, 1), (0,)], he=he),
    "two_cells_apart": lambda he: _thin(_walled([(0, 1), (0,)], he=he), 2),
    "three_cells_apart": lambda he: _thin(_walled([(0, 1, 2), (0,)], he=he), 3),
    # walls that meet, on blocks glued along the line where they do
    "cut": lambda he: cases.split_block_case(_walled([(0, 2)], blocks=((12, 9, 10),), he=he), ((12,), (4, 5), (4, 6))),
}


@pytest.mark.parametrize("he", [False, True])
@pytest.mark.parametrize("walls", list(WALLS))
def test_sync_where_walls_meet(oracle_mod, walls, he):
    """The wall states of random values, face after face: a later face reads what an
    earlier one has set, and the blocks behind such a block get theirs too."""
    case = WALLS[walls](he)
    print(f"[case] walls {walls} he={he} dims={[b.dims for b in case.blocks]}", flush=True)
    rng = np.random.default_rng(8)
    g = Mercury(case)
    o = oracle_mod.Oracle(case)
    try:
        names = ["U_H", "U_Na", "J_cell"] + (["U_He"] if he else [])
        for name in names:
            for ib in range(case.nb):
                v = rng.uniform(0.1, 2.0, (field_info(name)[1],) + case.box(ib))
                g.set(name, ib, v)
                o.set(name, ib, v)
        for op in ("sync_ucell", "sync_jcell"):
            g.op(op)
            o.op(op, 0)
        for name in names:
            for ib in range(case.nb):
                np.testing.assert_array_equal(g.get(name, ib), o.get(name, ib), err_msg=f"{name}[{ib}]")
    finally:
        g.close()


def test_steps_between_walls_that_meet(oracle_mod):
    case = WALLS["adjacent"](False)
    g = Mercury(case)
    o = oracle_mod.Oracle(case)
    try:
        g.prepare()
        o.prepare()
        np.testing.assert_array_equal(g.step(2), o.step(2))
        for name in ("U_H", "U_Na", "B_xi", "B_eta", "B_zeta", "J_cell"):
            for ib in range(case.nb):
                np.testing.assert_array_equal(g.get(name, ib), o.get(name, ib), err_msg=f"{name}[{ib}]")
    finally:
        g.close()
