"""The damped quench with the next step queued ahead (small boxes) and without (large ones): a quench
that converges in its first step moves the atoms by that step alone, whatever was queued behind it;
one that does not stops after maxsteps with the corrector."""
import numpy as np
import pytest

import msmpscu_amd.configs as cfg
import msmpscu_amd.mdlib as md

pytestmark = pytest.mark.gpu


def _device(cells):
    box = cfg.make_bcc_box(cells, cfg.W_A, 0.05, 300.0, 21)
    ctrl = cfg.w_ctrl(mx=64)
    fc = md.MDForceClassGPU(ForceTable=cfg.w_forcetable(box, ctrl))
    md.Register_ForceClass("FS_TYPE", fc)
    md.Initialize_Globle_Variables_DEV([box], ctrl, fc)
    md.Init_Forcetable_Dev([box], ctrl, fc)
    fc.Device.build_neighbors()
    fc.Device.calc_force()
    return fc.Device, ctrl


@pytest.mark.parametrize("cells", [(5, 5, 5), (32, 32, 32), (32, 32, 33)])
@pytest.mark.parametrize("maxsteps,steps", [(0, 1), (1, 1), (9, 1), (2, 3)])
def test_first_steps(cells, maxsteps, steps):
    dev, ctrl = _device(cells)
    mindele = 1.0e3 if steps == 1 else -1.0
    got, _ = dev.dyn_damp(maxsteps, mindele, ctrl.H)
    assert got == steps
    x, v, f, _, dis = dev.get_atoms()
    dev.close()
    ref, _ = _device(cells)
    for k in range(min(maxsteps, 1) if steps == 1 else maxsteps):
        if k:
            ref.correction(ctrl.H)
        ref.damping()
        ref.predictor(ctrl.H)
        ref.calc_force()
    if steps > 1:
        ref.correction(ctrl.H)
    rx, rv, rf, _, rdis = ref.get_atoms()
    ref.close()
    # the same operations in the same order, forces from an energy pass's F' (1e-12 relative)
    assert np.max(np.abs(x - rx)) <= 1e-13
    assert np.max(np.abs(dis - rdis)) <= 1e-13
    assert np.max(np.abs(v - rv)) <= 1e-12 * np.max(np.abs(rv))
    assert np.max(np.abs(f - rf)) <= 1e-11 * np.max(np.abs(rf))
