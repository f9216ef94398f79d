"""The list-walk density, force, energy and stress passes against the oracle at the sizes where their lanes per
atom and table placement change (32, 16, 8 lanes with the global table, 8, 4, 2 with the knots in
LDS), and on positions whose pairs leave the fast road: atoms a box length or more out, pairs
closer than the LDS window reaches.  Bars: F' 1e-13, forces 1e-10 eV/A max-abs, total
energy 1e-12 relative, each atom's energy and stress 1e-13 of their largest absolute value (sums of
at most a hundred terms)."""
import numpy as np
import pytest

import msmpscu_amd.configs as cfg
import msmpscu_amd.mdlib as md

pytestmark = pytest.mark.gpu


def _case(name):
    kind, n = name.split("-")
    c = {"250": (5, 5, 5), "8k": (16, 16, 16), "16k": (20, 21, 19), "39k": (27, 27, 27),
         "130k": (40, 41, 40), "1k": (6, 6, 7), "41k": (21, 22, 22)}[n]
    if kind == "cuni":
        box = cfg.make_cuni_slab(c, 3.57, 900.0, 5)
        ctrl = cfg.cuni_ctrl()
        return box, ctrl, cfg.cuni_forcetable(box, ctrl), None
    box = cfg.make_bcc_box(c, cfg.W_A, 0.05, 300.0, 11, n_vac=2)
    ctrl = cfg.w_ctrl(mx=64)
    ft = cfg.w_forcetable(box, ctrl, pot_type="EAM_TYPE" if kind == "eam" else "FS_TYPE")
    xp = box.XP.copy()
    if kind == "far":
        # trial points: one box length out, several, on the far face, and two atoms 0.4 A apart
        xp[3] += box.ZL * [1.0, 0.0, 0.0]
        xp[40] -= box.ZL * [0.0, 3.25, 0.5]
        xp[box.NPRT // 2] = box.BOXLOW + 0.01
        xp[box.NPRT - 1] = xp[box.NPRT - 2] + [0.4, 0.0, 0.0]
    return box, ctrl, ft, xp if kind == "far" else None


@pytest.mark.parametrize("name", ["fs-250", "eam-8k", "fs-16k", "eam-39k", "fs-130k", "cuni-1k",
                                  "cuni-41k", "far-250", "far-16k", "far-39k"])
def test_walk_passes_vs_oracle(orc, name):
    box, ctrl, ft, trial = _case(name)
    fc = md.MDForceClassGPU(ForceTable=ft)
    md.Register_ForceClass(ft.PotType, fc)
    md.Initialize_Globle_Variables_DEV(box, ctrl, fc)
    md.Init_Forcetable_Dev(box, ctrl, fc)
    dev = fc.Device
    dev.build_neighbors()
    x = box.XP
    if trial is not None:
        dev.put_atoms(trial)
        x = trial
    dev.calc_force()
    it = box.ITYP - 1
    kv, ind = orc.nlist("full", box.XP, it, box.STATU, box.BOXLOW, box.ZL, ctrl.IFPD, ctrl.NB_RM,
                        ctrl.NB_MXNBS)
    ru2, t = float(np.max(ctrl.RU)) ** 2, orc.from_mdlib(ft)
    fo, do, eo = orc.force_full(np.asfortranarray(x), it, box.STATU, kv, ind, box.ZL, ctrl.IFPD,
                                ru2, t)
    ao, aabs = orc.atomic_stress_full(np.asfortranarray(x), it, box.STATU, kv, ind, box.ZL,
                                      ctrl.IFPD, ru2, t, do, with_abs=True)
    df = np.max(np.abs(dev.get_forces() - fo))
    dd = np.max(np.abs(dev.get_den() - do) / np.maximum(1.0, np.abs(do)))
    dev.calc_epot()
    de = np.max(np.abs(dev.get_epot() - eo)) / np.max(np.abs(eo))
    et = abs(dev.get_box_epot()[0] - eo.sum()) / abs(eo.sum())
    da = np.max(np.abs(dev.calc_atomic_stress() - ao)) / np.max(aabs)
    print(f"{name}: n={box.NPRT} {dev.pass_kernel()} max|dF|={df:.3e} max|dF'|={dd:.3e} "
          f"dE {de:.3e} total {et:.3e} stress {da:.3e}")
    dev.close()
    assert df <= 1e-10
    assert dd <= 1e-13
    assert de <= 1e-13 and et <= 1e-12
    assert da <= 1e-13


@pytest.mark.parametrize("name", ["fs-250", "eam-8k", "fs-16k", "eam-39k", "fs-130k", "cuni-1k",
                                  "cuni-41k"])
def test_lost_atoms_leave_their_neighbours_alone(orc, name):
    """Atoms that went to NaN, infinity or 1e200 A since the list was built are outside every cutoff:
    energies and stresses of the others, the forces that come with them, and those of the force pass
    with a global table are those of the sums without them."""
    box, ctrl, ft, _ = _case(name)
    fc = md.MDForceClassGPU(ForceTable=ft)
    md.Register_ForceClass(ft.PotType, fc)
    md.Initialize_Globle_Variables_DEV(box, ctrl, fc)
    md.Init_Forcetable_Dev(box, ctrl, fc)
    dev = fc.Device
    dev.build_neighbors()
    x = box.XP.copy()
    lost = [7, 100, 150, 201]
    x[7, 0] = np.nan
    x[100] = [np.inf, 0.0, -np.inf]
    x[150, 2] = 1e200
    x[201] = np.nan
    dev.put_atoms(x)
    it = box.ITYP - 1
    kv, ind = orc.nlist("full", box.XP, it, box.STATU, box.BOXLOW, box.ZL, ctrl.IFPD, ctrl.NB_RM,
                        ctrl.NB_MXNBS)
    ru2, t = float(np.max(ctrl.RU)) ** 2, orc.from_mdlib(ft)
    fo, do, eo = orc.force_full(np.asfortranarray(x), it, box.STATU, kv, ind, box.ZL, ctrl.IFPD,
                                ru2, t)
    ao, aabs = orc.atomic_stress_full(np.asfortranarray(x), it, box.STATU, kv, ind, box.ZL,
                                      ctrl.IFPD, ru2, t, do, with_abs=True)
    rest = np.setdiff1d(np.arange(box.NPRT), lost)
    assert np.isfinite(fo[rest]).all() and np.isfinite(ao[rest]).all()
    dev.calc_epot()
    e = dev.get_epot()[rest]
    dev.calc_force()
    f, d = dev.get_forces()[rest], dev.get_den()[rest]
    a = dev.calc_atomic_stress()[rest]
    fs = dev.get_forces()[rest]
    if dev.pass_kernel() == "lds_table":
        f = fs
    dev.close()
    bad = {k: int(np.sum(~np.isfinite(v).reshape(len(rest), -1).all(axis=1)))
           for k, v in (("e", e), ("f", f), ("d", d), ("stress", a), ("f of stress", fs))}
    print(f"{name}: n={box.NPRT} not finite {bad}")
    assert not any(bad.values()), bad
    assert np.max(np.abs(f - fo[rest])) <= 1e-10 and np.max(np.abs(fs - fo[rest])) <= 1e-10
    assert np.max(np.abs(d - do[rest]) / np.maximum(1.0, np.abs(do[rest]))) <= 1e-13
    assert np.max(np.abs(e - eo[rest])) <= 1e-13 * np.max(np.abs(eo[rest]))
    assert np.max(np.abs(a - ao[rest])) <= 1e-13 * np.max(aabs[rest])


@pytest.mark.parametrize("name", ["eam-39k", "fs-130k", "cuni-41k"])
def test_pairs_at_the_edge_of_the_window(orc, name):
    """Hundreds of pairs at the distance where the knots in LDS begin (three eighths of the table),
    as near to it as coordinates go, in all directions: each counts once, on whichever side of the edge
    rounding puts it.  Bars as above, relative to the largest absolute value."""
    box, ctrl, ft, _ = _case(name)
    rng = np.random.default_rng(17)
    edge = 3 * ((ft.NTAB + 2) // 8) / ft.CSI
    r = edge * edge
    x = box.XP.copy()
    fc = md.MDForceClassGPU(ForceTable=ft)
    md.Register_ForceClass(ft.PotType, fc)
    md.Initialize_Globle_Variables_DEV(box, ctrl, fc)
    md.Init_Forcetable_Dev(box, ctrl, fc)
    dev = fc.Device
    dev.build_neighbors()
    kv, ind = dev.get_neighbors()
    used = np.zeros(box.NPRT, dtype=bool)
    inside = np.all((x - box.BOXLOW > 1.0) & (box.BOXLOW + box.ZL - x > 1.0), axis=1)
    pairs = 0
    for i in range(box.NPRT):
        js = ind[i, :kv[i]] - 1
        if pairs == 3000 or used[i] or not inside[i] or not kv[i] or used[js].any():
            continue
        j = js[np.argmin(np.sum((box.XP[js] - box.XP[i]) ** 2, axis=1))]
        d = rng.normal(size=3)
        x[j] = x[i] + d * (r / np.linalg.norm(d))
        used[js] = used[i] = True
        pairs += 1
    assert pairs > 100
    dev.put_atoms(x)
    it = box.ITYP - 1
    okv, oind = orc.nlist("full", box.XP, it, box.STATU, box.BOXLOW, box.ZL, ctrl.IFPD, ctrl.NB_RM,
                          ctrl.NB_MXNBS)
    ru2, t = float(np.max(ctrl.RU)) ** 2, orc.from_mdlib(ft)
    fo, do, eo = orc.force_full(np.asfortranarray(x), it, box.STATU, okv, oind, box.ZL, ctrl.IFPD,
                                ru2, t)
    ao, aabs = orc.atomic_stress_full(np.asfortranarray(x), it, box.STATU, okv, oind, box.ZL,
                                      ctrl.IFPD, ru2, t, do, with_abs=True)
    dev.calc_force()
    f, d = dev.get_forces(), dev.get_den()
    dev.calc_epot()
    e, a = dev.get_epot(), dev.calc_atomic_stress()
    dev.close()
    err = [np.max(np.abs(f - fo)) / np.max(np.abs(fo)), np.max(np.abs(d - do)) / np.max(np.abs(do)),
           np.max(np.abs(e - eo)) / np.max(np.abs(eo)), np.max(np.abs(a - ao)) / np.max(aabs)]
    print(f"{name}: {pairs} pairs at {r:.4f} A, force up to {np.max(np.abs(fo)):.3g}, errors "
          + " ".join(f"{v:.2e}" for v in err))
    assert err[0] <= 1e-12 and err[1] <= 1e-13 and err[2] <= 1e-13 and err[3] <= 1e-12
