"""Copies to and from the caller's arrays: up to 64 KB through the context's pinned words, to the host
beyond 4 MB through the shared ring in chunks and up to half a megabyte, where it is several arrays,
through one slot of it, else plain.  Sizes around these lines, and over several
rounds of the ring; several contexts at once.  Values come back bit for bit."""
import threading

import numpy as np
import pytest

import msmpscu_amd.configs as cfg
import msmpscu_amd.mdlib as md

pytestmark = pytest.mark.gpu


def _device(cells, seed):
    box = cfg.make_bcc_box(cells, cfg.W_A, 0.05, 300.0, seed)
    ctrl = cfg.w_ctrl(mx=64)
    fc = md.MDForceClassGPU(ForceTable=cfg.w_forcetable(box, ctrl))
    md.Register_ForceClass("FS_TYPE", fc)
    md.Initialize_Globle_Variables_DEV([box], ctrl, fc)
    md.Init_Forcetable_Dev([box], ctrl, fc)
    fc.Device.build_neighbors()      # cell order
    return fc.Device, box


def _round_trip(cells, seed):
    dev, box = _device(cells, seed)
    n = box.NPRT
    rng = np.random.default_rng(seed)
    x = box.XP + rng.uniform(-0.01, 0.01, (n, 3))
    x = box.BOXLOW + np.mod(x - box.BOXLOW, box.ZL)     # still inside the box
    v, d = rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    dev.put_atoms(x, v)
    dev.put_dis(d)
    xp, xp1, fp, st, dis = dev.get_atoms()
    ok = all(np.array_equal(a, b) for a, b in ((xp, x), (xp1, v), (dis, d), (st, box.STATU)))
    ok = ok and np.array_equal(dev.get_forces(), fp)
    e = rng.normal(size=n)
    dev.build_neighbors()
    dev.calc_epot()
    e0 = dev.get_epot()
    dev.add_epot(e)
    ok = ok and np.array_equal(dev.get_epot(), e0 + e)
    dev.put_atoms(None, x)
    ok = ok and np.array_equal(dev.get_atoms()[1], x)
    kv, ind = dev.get_neighbors()
    ok = ok and kv.shape == (n,) and ind.shape[0] == n and kv.min() > 0
    dev.close()
    return ok


# 2 * product atoms: one array of 3 n doubles is 64 KB at 2730.7 atoms, all five 104 n at 630.2
@pytest.mark.parametrize("cells", [(4, 4, 4), (5, 7, 9), (3, 5, 21), (7, 13, 15), (5, 21, 13),
                                   (21, 26, 40), (41, 41, 42), (26, 27, 29), (27, 27, 29),
                                   (13, 14, 14), (14, 14, 14)])
def test_round_trip(cells):
    assert _round_trip(cells, 5)


def test_contexts_at_once():
    res = {}

    def work(k, cells):
        res[k] = all(_round_trip(cells, 10 * k + j) for j in range(3))
    th = [threading.Thread(target=work, args=(k, c))
          for k, c in enumerate([(4, 4, 4), (21, 26, 40), (20, 30, 30), (7, 13, 15)])]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert res == {k: True for k in range(4)}
