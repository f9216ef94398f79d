"""The wave-per-cell list and the cell sort where they can go wrong: both sort paths (one workgroup
up to 8192 atoms), more than 64 atoms in a cell, more candidates around a cell than one chunk
holds, out-of-box atoms, list radii that differ between species, several boxes.  The list must
equal the per-atom scan's entry for entry, and the oracle's as sets."""
import numpy as np
import pytest

import msmpscu_amd._lib as L
import msmpscu_amd.configs as cfg
import msmpscu_amd.mdlib as md

pytestmark = pytest.mark.gpu


def _device(boxes, ctrl, ft, mode):
    fc = md.MDForceClassGPU(ForceTable=ft)
    md.Register_ForceClass(ft.PotType, fc)
    md.Initialize_Globle_Variables_DEV(boxes, ctrl, fc)
    md.Init_Forcetable_Dev(boxes, ctrl, fc)
    fc.Device.set_option(L.MSM_OPT_NLIST_KERNEL, mode)
    return fc.Device


def _case(name):
    ctrl = cfg.w_ctrl(mx=64)
    if name == "crowd":   # 70 atoms in one cell
        box = cfg.make_bcc_box((6, 6, 6), cfg.W_A, 0.03, 0.0, 4)
        x = np.concatenate([box.XP, np.random.default_rng(4).uniform(0.1, 2.2, (70, 3))])
        n = x.shape[0]
        box = md.SimMDBox(NPRT=n, NGROUP=1, ZL=box.ZL, BOXLOW=box.BOXLOW, XP=np.asfortranarray(x),
                          XP1=np.zeros((n, 3)), ITYP=np.ones(n, np.int32),
                          STATU=np.ones(n, np.int32), CM=box.CM, PTYPE=box.PTYPE)
        ctrl = cfg.w_ctrl(mx=200)
        return [box], ctrl, cfg.w_forcetable(box, ctrl)
    if name == "radii":
        box = cfg.make_cuni_slab((6, 7, 6), 3.57, 300.0, 9)
        ctrl = cfg.cuni_ctrl()
        ctrl.NB_RM = np.asfortranarray([[6.3, 5.9], [5.9, 6.1]])
        return [box], ctrl, cfg.cuni_forcetable(box, ctrl)
    if name == "boxes":
        boxes = [cfg.make_bcc_box(c, cfg.W_A, 0.05, 300.0, k, n_vac=k)
                 for k, c in enumerate([(5, 6, 7), (15, 16, 17), (3, 4, 9)])]
        return boxes, ctrl, cfg.w_forcetable(boxes[0], ctrl)
    cells = {"8190": (16, 16, 16), "8194": (16, 16, 17), "outside": (9, 9, 9)}[name]
    box = cfg.make_bcc_box(cells, cfg.W_A, 0.05, 300.0, 3)
    if name == "outside":
        st = box.STATU.copy()
        st[[5, 700]] = md.CP_STATU_ACTIVE | md.CP_STATU_OUTOFBOX
        box.STATU = st
        box.XP[5] = box.BOXLOW - 3.0
    return [box], ctrl, cfg.w_forcetable(box, ctrl)


@pytest.mark.parametrize("name", ["8190", "8194", "crowd", "outside", "radii", "boxes"])
def test_cell_list_equals_scan(orc, name):
    boxes, ctrl, ft = _case(name)
    got = []
    for mode in (0, 1):
        dev = _device(boxes, ctrl, ft, mode)
        dev.build_neighbors()
        dev.build_neighbors()      # from cell order too
        got.append(dev.get_neighbors())
        dev.close()
    (kv, ind), (kv1, ind1) = got
    print(f"{name}: n={len(kv)} longest {kv.max()}")
    assert np.array_equal(kv, kv1)
    live = np.arange(ind.shape[1])[None, :] < kv[:, None]
    assert np.array_equal(np.where(live, ind, 0), np.where(live, ind1, 0))
    off = 0
    for b in boxes:
        okv, oind = orc.nlist("full", b.XP, b.ITYP - 1, b.STATU, b.BOXLOW, b.ZL, ctrl.IFPD,
                              ctrl.NB_RM, ctrl.NB_MXNBS)
        assert np.array_equal(kv[off:off + b.NPRT], okv)
        for i in range(b.NPRT):
            mine = np.sort(ind[off + i, : okv[i]]) - 1 - off
            assert np.array_equal(mine, np.sort(oind[i, : okv[i]]))
        off += b.NPRT
