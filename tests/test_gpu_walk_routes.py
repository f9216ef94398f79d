"""Which kernel runs, and that it is right there: the list walk's lanes and table placement at the sizes
where the rule for them changes, the shapes that only large systems take (one lane an atom on several
boxes, four on alloys, alloys with tables too large for the LDS), and the kernels with 64-bit offsets
that take over from the walk's atom limit on.  Density, forces, energies and stresses against the
oracle, with the bars of test_gpu_walk.py."""
import numpy as np
import pytest

import msmpscu_amd._lib as L
import msmpscu_amd.configs as cfg
import msmpscu_amd.mdlib as md

pytestmark = pytest.mark.gpu


def _device(boxes, ctrl, ft):
    fc = md.MDForceClassGPU(ForceTable=ft)
    md.Register_ForceClass(ft.PotType, fc)
    md.Initialize_Globle_Variables_DEV(boxes, ctrl, fc)
    md.Init_Forcetable_Dev(boxes, ctrl, fc)
    return fc.Device


def _check(orc, dev, boxes, ctrl, ft, steps=0):
    """The passes on the current positions, after a run of some steps (whose last forces are those of the
    lists it ends with: an atom may have come into reach since they were built)."""
    dev.build_neighbors()
    if steps:
        dev.calc_force()
        dev.run(steps, ctrl.NB_UPTAB, 0, ctrl.H)
        run_f = dev.get_forces()
        run_kv, run_ind = dev.get_neighbors()
    x = dev.get_atoms()[0]
    dev.build_neighbors()
    dev.calc_force()
    f, d = dev.get_forces(), dev.get_den()
    dev.calc_epot()
    e, eb = dev.get_epot(), dev.get_box_epot()
    s = dev.calc_atomic_stress()
    ru2, t, off = float(np.max(ctrl.RU)) ** 2, orc.from_mdlib(ft), 0
    worst = np.zeros(5)
    for b, box in enumerate(boxes):
        n, it = box.NPRT, box.ITYP - 1
        w = slice(off, off + n)
        off += n
        xb = np.asfortranarray(x[w])
        kv, ind = orc.nlist("full", xb, it, box.STATU, box.BOXLOW, box.ZL, ctrl.IFPD, ctrl.NB_RM,
                            ctrl.NB_MXNBS)
        fo, do, eo = orc.force_full(xb, it, box.STATU, kv, ind, box.ZL, ctrl.IFPD, ru2, t)
        so, sabs = orc.atomic_stress_full(xb, it, box.STATU, kv, ind, box.ZL, ctrl.IFPD, ru2, t, do,
                                          with_abs=True)
        if steps:
            rind = np.where(np.arange(run_ind.shape[1]) < run_kv[w, None], run_ind[w] - 1 - w.start, 0)
            ro, _, _ = orc.force_full(xb, it, box.STATU, run_kv[w], rind, box.ZL, ctrl.IFPD, ru2, t)
            dr = np.max(np.abs(run_f[w] - ro))
            assert dr <= 1e-10
        worst = np.maximum(worst, [
            np.max(np.abs(f[w] - fo)), np.max(np.abs(d[w] - do) / np.maximum(1.0, np.abs(do))),
            np.max(np.abs(e[w] - eo)) / np.max(np.abs(eo)), abs(eb[b] - eo.sum()) / abs(eo.sum()),
            np.max(np.abs(s[w] - so)) / np.max(sabs)])
    print(f"n={off} {dev.pass_kernel()} {dev.walk_lanes()} errors " + " ".join(f"{v:.2e}" for v in worst))
    assert worst[0] <= 1e-10 and worst[1] <= 1e-13 and worst[2] <= 1e-13
    assert worst[3] <= 1e-12 and worst[4] <= 1e-13


@pytest.mark.parametrize("kind,cells,kernel,lanes", [
    ("w", (5, 5, 5), "wide", 32), ("w", (16, 16, 16), "wide", 16), ("w", (20, 21, 19), "wide", 8),
    ("w", (27, 27, 27), "lds_table", 4), ("w", (40, 41, 40), "lds_table", 2),
    ("cuni", (6, 6, 7), "wide", 32), ("cuni", (21, 22, 22), "lds_table", 8)])
def test_lanes_and_table_follow_the_size(kind, cells, kernel, lanes):
    if kind == "cuni":
        box, ctrl = cfg.make_cuni_slab(cells, 3.57, 900.0, 5), cfg.cuni_ctrl()
        ft = cfg.cuni_forcetable(box, ctrl)
    else:
        box, ctrl = cfg.make_bcc_box(cells, cfg.W_A, 0.05, 300.0, 11, n_vac=2), cfg.w_ctrl(mx=64)
        ft = cfg.w_forcetable(box, ctrl)
    dev = _device([box], ctrl, ft)
    got = dev.pass_kernel(), dev.walk_lanes()
    dev.close()
    assert got == (kernel, (lanes, lanes))


@pytest.mark.parametrize("pot", ["FS_TYPE", "EAM_TYPE"])
def test_several_large_boxes(orc, pot):
    """203,546 atoms in two boxes: one lane an atom."""
    boxes = [cfg.make_bcc_box(c, cfg.W_A, 0.05, 300.0, 31 + k)
             for k, c in enumerate([(22, 22, 22), (45, 45, 45)])]
    ctrl = cfg.w_ctrl(mx=40)
    ft = cfg.w_forcetable(boxes[0], ctrl, pot_type=pot)
    dev = _device(boxes, ctrl, ft)
    assert dev.walk_lanes() == (1, 1) and dev.pass_kernel() == "lds_table"
    _check(orc, dev, boxes, ctrl, ft, steps=11)
    dev.close()


# atoms x neighbours below and above the line from which on a table that does not fit goes to the
# kernels without the walk; tables whose upper halves fit the LDS (5,000 knots) and do not (10,000: the
# density's does)
@pytest.mark.parametrize("cells,ntab,kernel,lanes", [
    ((25, 25, 25), 5000, "lds_table", (4, 4)), ((25, 25, 25), 10000, "wide", (4, 8)),
    ((31, 31, 31), 10000, "lanes", (4, 0))])
def test_alloy_tables(orc, cells, ntab, kernel, lanes):
    box = cfg.make_cuni_slab(cells, 3.57, 600.0, 7)
    ctrl = cfg.cuni_ctrl(ntab=ntab, mx=128)
    ft = cfg.cuni_forcetable(box, ctrl)
    dev = _device([box], ctrl, ft)
    assert (dev.pass_kernel(), dev.walk_lanes()) == (kernel, lanes)
    _check(orc, dev, [box], ctrl, ft, steps=6)
    dev.close()


def _limit_case(name):
    ctrl = cfg.w_ctrl(mx=64)
    if name == "boxes":
        boxes = [cfg.make_bcc_box(c, cfg.W_A, 0.05, 500.0, 30 + k, n_vac=k, n_dumbbell=k % 2)
                 for k, c in enumerate([(5, 6, 7), (9, 9, 9), (3, 4, 5)])]
        return boxes, ctrl, cfg.w_forcetable(boxes[0], ctrl)
    if name == "cuni":
        box = cfg.make_cuni_slab((6, 6, 6), 3.57, 600.0, 5)
        ctrl = cfg.cuni_ctrl()
        return [box], ctrl, cfg.cuni_forcetable(box, ctrl)
    if name == "short":     # lists up to the capacity, many empty
        box = cfg.make_bcc_box((10, 10, 10), cfg.W_A, 0.05, 300.0, 77, vacancy_frac=0.8)
        return [box], cfg.w_ctrl(mx=11), cfg.w_forcetable(box, ctrl)
    box = cfg.make_bcc_box((8, 8, 8), cfg.W_A, 0.05, 300.0, 77)
    if name == "window":    # knots below the window, with pairs there
        for i, frac in [(10, 0.55), (200, 0.5), (555, 0.58)]:
            box.XP[i] = box.XP[i] + frac * cfg.W_A / 2
        box.XP = np.asfortranarray(cfg.wrap_into(box.XP, box.BOXLOW, box.ZL, (1, 1, 1)))
        ctrl = cfg.w_ctrl(ntab=12000)
    return [box], ctrl, cfg.w_forcetable(box, ctrl, pot_type="EAM_TYPE" if name == "eam" else "FS_TYPE")


@pytest.mark.parametrize("path", [1, 2, 4])
@pytest.mark.parametrize("name", ["fs", "eam", "boxes", "cuni", "window", "short"])
def test_beyond_the_walk(orc, name, path):
    """From the atom limit on the passes with 64-bit offsets run: whole-table windows in LDS for
    densities and forces, the general energy and stress passes.  (The limit is lowered; at 2^27 atoms
    it is not for a test.)"""
    boxes, ctrl, ft = _limit_case(name)
    dev = _device(boxes, ctrl, ft)
    if path != 2:       # 2 is what the choice by size falls back to
        dev.set_option(L.MSM_OPT_FORCE_PATH, path)
    n = sum(b.NPRT for b in boxes)
    dev.set_option(L.MSM_OPT_WALK_ATOMS, n + 1)
    assert min(dev.walk_lanes()) > 0
    dev.set_option(L.MSM_OPT_WALK_ATOMS, n)
    assert (dev.pass_kernel(), dev.walk_lanes()) == ("lds_table", (0, 0))
    _check(orc, dev, boxes, ctrl, ft, steps=0 if name in ("window", "short") else 12)
    dev.close()
