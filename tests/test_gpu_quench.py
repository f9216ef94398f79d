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


@pytest.mark.parametrize("maxsteps", [1, 2, 5])
def test_several_boxes(maxsteps):
    """Three boxes at once (the quench's kernels read each atom's own box) against the same steps taken
    one by one, and against each box quenched alone."""
    boxes = [cfg.make_bcc_box(c, cfg.W_A, 0.08, 600.0, 40 + k, n_vac=k)
             for k, c in enumerate([(5, 5, 5), (9, 8, 7), (3, 4, 5)])]
    ctrl = cfg.w_ctrl(mx=64)

    def device(bs):
        fc = md.MDForceClassGPU(ForceTable=cfg.w_forcetable(boxes[0], ctrl))
        md.Register_ForceClass("FS_TYPE", fc)
        md.Initialize_Globle_Variables_DEV(bs, ctrl, fc)
        md.Init_Forcetable_Dev(bs, ctrl, fc)
        fc.Device.build_neighbors()
        fc.Device.calc_force()
        return fc.Device

    def quenched(bs):
        dev = device(bs)
        assert dev.dyn_damp(maxsteps, -1.0, ctrl.H)[0] == maxsteps + 1
        x, v, f, _, dis = dev.get_atoms()
        dev.close()
        return x, v, f, dis

    got = quenched(boxes)
    alone = [np.concatenate(a) for a in zip(*(quenched([b]) for b in boxes))]
    ref = device(boxes)
    for k in range(maxsteps):
        if k:
            ref.correction(ctrl.H)
        ref.damping()
        ref.predictor(ctrl.H)
        ref.calc_force()
    ref.correction(ctrl.H)
    x, v, f, _, dis = ref.get_atoms()
    ref.close()
    for other in (alone, (x, v, f, dis)):
        for a, b, bar in zip(got, other, (1e-13, 1e-12 * np.max(np.abs(v)), 1e-11 * np.max(np.abs(f)),
                                          1e-13)):
            assert np.max(np.abs(a - b)) <= bar
