"""Halo plans and alias classes supplied by the caller (MERCURY_BC_EXTERNAL faces).

A context whose block connections are EXTERNAL faces knows no neighbour there;
the caller uploads the halo and owner -> alias copies of every sync group
(mercury_set_sync_plan) and the alias-mean classes of the shared edges
(mercury_set_alias_classes), together with the ghost geometry its own topology
code computes.  Here the plans, classes and geometry are those the library
builds for the same blocks glued by interfaces (read back with
mercury_sync_plan / mercury_alias_classes), so the two contexts must step bit
for bit alike in every form and from a captured graph.  A second test checks
the entry semantics on a hand-built plan with a sign flip and a component
swap, the two things a rotated or mirrored connection needs.
"""
import copy

import numpy as np
import pytest

from mpcns_mercury_amd import cases
from mpcns_mercury_amd.hip import Mercury, MercuryError, field_info

pytestmark = pytest.mark.gpu

GROUPS = ["Ucell", "Bface", "Eedge", "Ehall", "Jedge", "B_cell", "J_cell", "Badd", "Eres", "Eres0", "dB"]
GEOM = ["Jac", "JDxi", "JDet", "JDze", "Area_xi", "Area_eta", "Area_zeta", "beta_xi", "beta_eta", "beta_zeta",
        "dl_xi", "dl_eta", "dl_zeta", "alpha_xi", "alpha_eta", "alpha_zeta", "dr_xi", "dr_eta", "dr_zeta",
        "Bcell_from_Bface_w", "Jcell_from_Jedge_w", "cell_center", "taper_xi", "taper_eta", "taper_zeta",
        "eta_local_xi", "eta_local_eta", "eta_local_zeta"]
INPUTS = ["U_H", "U_Na", "B_xi", "B_eta", "B_zeta", "Badd_xi", "Badd_eta", "Badd_zeta"]
CHECK = ["U_H", "U_Na", "B_xi", "B_eta", "B_zeta", "B_cell", "J_cell", "J_xi", "J_eta", "J_zeta", "E_xi", "PV_H", "U_plus"]


def _external(case):
    c = copy.deepcopy(case)
    for b in c.blocks:
        b.bc = tuple(cases.BC_EXTERNAL if x == cases.BC_INTERFACE else x for x in b.bc)
        b.nbr = (-1,) * 6
        b.off = ((0, 0, 0),) * 6
    return c


def _same(ga, gb, case, ctx):
    for ib in range(case.nb):
        for name in CHECK:
            np.testing.assert_array_equal(gb.get(name, ib), ga.get(name, ib), err_msg=f"{ctx}: {name}[{ib}]")


@pytest.mark.parametrize("form", [0, 1, 2])
def test_caller_plans_reproduce_the_interfaces(form):
    a = cases.make_split_cube(n=(12, 10, 8), split=(2, 2, 1), hall=True)
    b = _external(a)
    print(f"[case] {a.name}: interfaces as EXTERNAL faces with the interface plans, form {form}", flush=True)
    ga, gb = Mercury(a), Mercury(b)
    try:
        for ib in range(a.nb):
            for name in GEOM + INPUTS:
                gb.set(name, ib, ga.get(name, ib))
        n_copies = 0
        for grp in GROUPS:
            for stage in (0, 1):
                plan = ga.sync_plan(grp, stage)
                n_copies += len(plan)
                gb.set_sync_plan(grp, stage, plan)
                np.testing.assert_array_equal(gb.sync_plan(grp, stage), plan)
        assert n_copies > 0
        classes = ga.alias_classes()
        assert len(classes[1]) > 0
        gb.set_alias_classes(*classes)
        for x, y in zip(gb.alias_classes(), classes):
            np.testing.assert_array_equal(x, y)
        for g in (ga, gb):
            g.prepare()
            g.set_form(form)
        np.testing.assert_array_equal(gb.step(3, 0), ga.step(3, 0))
        _same(ga, gb, a, "3 steps")
        if form >= 1:
            for g in (ga, gb):
                g.graph_capture(1)
                g.graph_launch(2)
                g.synchronize()
            _same(ga, gb, a, "graph replay, RK2")
    finally:
        ga.close()
        gb.close()


def test_plan_entry_semantics_and_refusals():
    """dst = sign * src across components and blocks, after the group's own copies."""
    case = _external(cases.make_split_cube(n=(8, 8, 6), split=(2, 1, 1)))
    g = Mercury(case)
    try:
        sx, _, _ = field_info("B_xi")
        sy, _, _ = field_info("B_eta")
        # the first ghost face beyond block 0's -xi face takes minus block 1's
        # eta flux at a chosen owned face, as a mirrored, rotated connection would
        rng = np.random.default_rng(3)
        vals = rng.standard_normal((case.nb,) + case.box(0))
        for ib in range(case.nb):
            g.set("B_eta", ib, vals[ib])
        g.set_sync_plan("Bface", 0, [[sx, 0, -1, 2, 3, sy, 1, 5, 4, 2, -1], [sx, 0, -1, 3, 3, sy, 1, 5, 5, 2, 1]])
        g.op("sync_bface")
        got = g.get("B_xi", 0)[0]
        gg = case.g
        after = g.get("B_eta", 1)[0]
        assert got[gg - 1, gg + 2, gg + 3] == -after[gg + 5, gg + 4, gg + 2]
        assert got[gg - 1, gg + 3, gg + 3] == after[gg + 5, gg + 5, gg + 2]
        with pytest.raises(MercuryError, match="outside the block's box"):
            g.set_sync_plan("Bface", 0, [[sx, 0, -gg - 1, 0, 0, sy, 1, 0, 0, 0, 1]])
        with pytest.raises(MercuryError, match="sign must be"):
            g.set_sync_plan("Bface", 0, [[sx, 0, 0, 0, 0, sy, 1, 0, 0, 0, 2]])
        with pytest.raises(MercuryError, match="unknown sync group"):
            g.set_sync_plan("Bfaces", 0, [])
    finally:
        g.close()


# every length that a joined plan can hold in a wave, one more, and one that spans workgroups
@pytest.mark.parametrize("lengths", [(1, 2, 3, 4, 5), (63, 1, 62, 2, 64), (65,), (300, 2, 64)])
def test_joined_plans_read_before_they_write(lengths):
    """Random plans of both stages on the groups of a pair, with chains (an entry
    reads what the next one writes), cycles, signs, components and blocks mixed, and
    owner entries that read and replace what the halo stage wrote: each plan acts as
    one gather and one scatter, in the order halo stages, owner stages.  Bit for bit
    (copies and sign flips)."""
    case = _external(cases.make_split_cube(n=(12, 12, 10), split=(2, 1, 1)))
    print(f"[case] joined plans, chains of {lengths}", flush=True)
    rng = np.random.default_rng(sum(lengths))
    box, gg = case.box(0), case.g
    groups = {"Ucell": [("U_H", c) for c in range(5)] + [("U_Na", c) for c in range(5)], "Bface": [(f"B_{a}", 0) for a in ("xi", "eta", "zeta")]}
    start = {n: rng.standard_normal((case.nb, field_info(n)[1]) + box) for n in {n for v in groups.values() for n, _ in v}}

    def point(name, c):
        # owned cells of both blocks, faces with them
        return (name, c, int(rng.integers(case.nb))) + tuple(int(rng.integers(0, m - 2 * gg - 1)) for m in box)

    def row(d, s, sign):
        return [field_info(d[0])[0] + d[1], *d[2:], field_info(s[0])[0] + s[1], *s[2:], sign]

    plans = {}
    for grp, comps in groups.items():
        pick = lambda: point(*comps[int(rng.integers(len(comps)))])  # noqa: E731
        seen, halo = set(), []

        def fresh():
            p = pick()
            while p in seen:
                p = pick()
            seen.add(p)
            return p

        for n in lengths:
            pts = [fresh() for _ in range(n + 1)]
            if n > 2 and n % 2:
                pts[n] = pts[0]  # a cycle
            halo += [(pts[i], pts[i + 1], int(rng.choice([-1, 1]))) for i in range(n)]
        halo += [(fresh(), fresh(), 1) for _ in range(150)]
        halo = [halo[i] for i in rng.permutation(len(halo))]
        # an owner entry replaces a halo value, reads one, or neither
        owner = [(halo[i][0], fresh(), -1) for i in range(0, 20)] + [(fresh(), halo[i][0], -1) for i in range(20, 40)]
        owner += [(halo[i][0], halo[i + 20][0], 1) for i in range(40, 60)] + [(fresh(), fresh(), -1) for _ in range(70)]
        plans[grp] = (halo, owner)

    def run(with_plans):
        g = Mercury(case)
        try:
            for grp, stages in plans.items():
                for t in (0, 1):
                    g.set_sync_plan(grp, t, [row(*e) for e in stages[t]] if with_plans else np.zeros((0, 11), np.int32))
            for n, v in start.items():
                for ib in range(case.nb):
                    g.set(n, ib, v[ib])
            g.op("sync_ucell")
            g.op("sync_bface")
            return {n: np.stack([g.get(n, ib) for ib in range(case.nb)]) for n in start}
        finally:
            g.close()

    want, got = run(False), run(True)
    at = lambda p: (p[2], p[1], p[3] + gg, p[4] + gg, p[5] + gg)  # noqa: E731
    for stages in plans.values():
        for plan in stages:
            vals = [sign * want[s[0]][at(s)] for _, s, sign in plan]
            for (d, _, _), v in zip(plan, vals):
                want[d[0]][at(d)] = v
    for n in start:
        np.testing.assert_array_equal(got[n], want[n], err_msg=n)


def test_plans_set_one_by_one_and_again():
    """Each call plans only what it changes: plans set stage by stage with syncs in
    between, replaced, and set in another order leave every group's sync (those of
    the resistive correction, which this context has no program for at first, among
    them) as a context that gets the last plans only."""
    a = cases.make_split_cube(n=(12, 10, 8), split=(2, 2, 1), hall=True)
    b = _external(a)
    print("[case] caller plans one by one", flush=True)
    ops = {"Ucell": "sync_ucell", "Bface": "sync_bface", "Eedge": "sync_eedge", "Ehall": "sync_ehall", "Jedge": "sync_jedge",
           "B_cell": "sync_bcell", "J_cell": "sync_jcell", "Badd": "sync_badd", "Eres": "sync_eres", "dB": "sync_db"}
    ga, gb, gc = Mercury(a), Mercury(b), Mercury(b)
    try:
        plans = {(grp, t): ga.sync_plan(grp, t) for grp in ops for t in (0, 1)}
        for k, p in plans.items():
            gc.set_sync_plan(*k, p)
        rng = np.random.default_rng(4)
        for n, (grp, t) in enumerate(sorted(plans, key=lambda k: (-k[1], k[0]))):
            gb.set_sync_plan(grp, t, plans[grp, t][::3])
            for op in list(ops.values())[n % 5::5]:
                gb.op(op)
        for k in reversed(plans):
            gb.set_sync_plan(*k, plans[k])
        names = INPUTS + ["E_xi", "E_eta", "E_zeta", "Ehall_xi", "Ehall_eta", "Ehall_zeta", "J_xi", "J_eta", "J_zeta", "B_cell", "J_cell",
                          "Eres_xi", "Eres_eta", "Eres_zeta", "dB_xi", "dB_eta", "dB_zeta"]
        for n in names:
            for ib in range(b.nb):
                v = rng.uniform(0.1, 2.0, (field_info(n)[1],) + b.box(ib))
                gb.set(n, ib, v)
                gc.set(n, ib, v)
        for op in ops.values():
            gb.op(op)
            gc.op(op)
        for n in names:
            for ib in range(b.nb):
                np.testing.assert_array_equal(gb.get(n, ib), gc.get(n, ib), err_msg=f"{n}[{ib}]")
    finally:
        for g in (ga, gb, gc):
            g.close()
