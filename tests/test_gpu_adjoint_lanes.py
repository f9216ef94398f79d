"""The adjoint passes with 4 and with 2 lanes an atom (more where the atoms are fewer, as in
test_gpu_adjoint.py): knot gradients against the oracle's adjoint at the smallest sizes that take
them, to the same 1e-10 of the largest entry."""
import numpy as np
import pytest

import msmpscu_amd.configs as cfg
import msmpscu_amd.mdlib as md
from msmpscu_amd import adjoint as adj

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(32, 32, 33), (40, 40, 41)])
def test_adjoint_lanes_match_oracle(orc, cells):
    ctrl = cfg.w_ctrl(mx=64)
    box = cfg.make_bcc_box(cells, cfg.W_A, 0.1, 300.0, 40, n_vac=3)
    box.STATU[[7, 100]] = 0
    ft = cfg.w_forcetable(box, ctrl, pot_type="EAM_TYPE")
    fc = md.MDForceClassGPU(ForceTable=ft)
    md.Register_ForceClass(ft.PotType, fc)
    md.Initialize_Globle_Variables_DEV([box], ctrl, fc)
    md.Init_Forcetable_Dev([box], ctrl, fc)
    dev = fc.Device
    dev.build_neighbors()
    G = np.random.default_rng(8).normal(size=(box.NPRT, 3))
    got = adj.table_grads(dev, G, np.array([0.7]), ft.NTAB, ft.NEMBD, True)
    dev.close()
    it = box.ITYP - 1
    kv, ind = orc.nlist("full", box.XP, it, box.STATU, box.BOXLOW, box.ZL, ctrl.IFPD, ctrl.NB_RM,
                        ctrl.NB_MXNBS)
    ref = orc.adjoint_full(box.XP, it, box.STATU, kv, ind, box.ZL, ctrl.IFPD,
                           float(np.max(ctrl.RU)) ** 2, orc.from_mdlib(ft), G, 0.7, None)
    for name in ("POTR", "FPOTR", "POTB", "FPOTB", "FEMBD", "DFEMBD"):
        r = ref[name.lower()][0, 1:-1]
        assert np.max(np.abs(got[name] - r)) <= 1e-10 * np.max(np.abs(r)), name
