"""The C-ABI's host paths on a runtime of host memory whose kernels do nothing (fake_hip.c): what a
call reports when a launch or an allocation fails.  Each case runs in a process of its own, since the
runtime has to be loaded before the library."""
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CASES = {}


def case(f):
    CASES[f.__name__] = f
    return f


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "fake_hip.c"),
                    "-lpthread"], check=True)
    return so


def _device(cells=(5, 5, 5), nbox=1):
    import msmpscu_amd.configs as cfg
    import msmpscu_amd.mdlib as md
    boxes = [cfg.make_bcc_box(cells, cfg.W_A, 0.05, 300.0, 3 + k) for k in range(nbox)]
    ctrl = cfg.w_ctrl(mx=32)
    fc = md.MDForceClassGPU(ForceTable=cfg.w_forcetable(boxes[0], ctrl))
    md.Register_ForceClass("FS_TYPE", fc)
    md.Initialize_Globle_Variables_DEV(boxes, ctrl, fc)
    md.Init_Forcetable_Dev(boxes, ctrl, fc)
    return fc.Device, boxes, ctrl


def _hip_error(call):
    try:
        call()
    except RuntimeError as e:
        assert "MSM_ERR_HIP" in str(e), e
        return True
    return False


@case
def refused_copies(f):
    """A copy whose kernel was not launched is an error, not the bytes of an earlier copy."""
    dev, boxes, _ = _device()
    x = np.array(boxes[0].XP)
    dev.get_atoms()
    f.fake_refuse(b"k_copy_words")
    assert _hip_error(dev.get_atoms)
    assert _hip_error(dev.get_epot)
    assert _hip_error(lambda: dev.put_atoms(x))
    assert _hip_error(lambda: dev.put_dis(x))
    dev.build_neighbors()
    f.fake_refuse(b"k_sum_chunks")
    assert _hip_error(dev.get_box_epot)
    f.fake_refuse(b"k_copy_out")
    assert _hip_error(dev.get_atoms)
    f.fake_refuse(b"k_sort_pos")
    assert _hip_error(lambda: dev.put_atoms(x))
    f.fake_refuse(b"")
    dev.get_atoms()     # and the error is not kept


@case
def refused_passes(f):
    """A call of which a kernel was not launched is an error; so is a quench whose step gives no
    note (here no kernel ever does)."""
    dev, _, ctrl = _device()
    dev.build_neighbors()
    for kernel, call in ((b"k_density", dev.calc_force), (b"k_force", dev.calc_force),
                         (b"k_energy", dev.calc_epot), (b"k_virial", dev.calc_atomic_stress),
                         (b"k_force", lambda: dev.run(2, ctrl.NB_UPTAB, 0, ctrl.H)),
                         (b"k_nlist", dev.build_neighbors),
                         (b"k_predictor", lambda: dev.dyn_damp(3, 0.0, ctrl.H)),
                         (b"k_damp_check", lambda: dev.dyn_damp(3, 0.0, ctrl.H))):
        f.fake_refuse(kernel)
        assert _hip_error(call), kernel
        f.fake_refuse(b"")
        dev.build_neighbors()
    dev.calc_force()
    dev.run(2, ctrl.NB_UPTAB, 0, ctrl.H)
    for maxsteps in (1, 2, 3):
        assert _hip_error(lambda: dev.dyn_damp(maxsteps, 0.0, ctrl.H))
    steps, _ = dev.dyn_damp(0, 0.0, ctrl.H)
    assert steps == 1


@case
def sort_buffers_after_failures(f):
    """The cell counts are zero when a rebuild starts: after a set_boxes that failed between its
    buffers, whatever grid the next one has, and after a rebuild of which a kernel was refused."""
    import ctypes as C

    import msmpscu_amd._lib as L
    dev, boxes, ctrl = _device((16, 16, 17))        # 8704 atoms: the sort of several launches
    box = boxes[0]

    def set_boxes(scale):
        n = np.array([box.NPRT], dtype=np.int32)
        lo, ln = np.array(box.BOXLOW, dtype=float), np.array(box.ZL, dtype=float) * scale
        return L.lib().msm_set_boxes(dev.h, 1, L.iptr(n), L.dptr(lo), L.dptr(ln),
                                     L.iptr(np.array([1, 1, 1], dtype=np.int32)))

    for k in (2, 3, 4):          # counts, starts, scan
        f.fake_dev_fail(k)
        assert set_boxes(2.0) == 3                          # MSM_ERR_NOMEM
        f.fake_dev_fail(0)
        assert L.lib().msm_build_neighbors(dev.h) == 7      # MSM_ERR_STATE: no boxes
        before = f.fake_memsets()
        assert set_boxes(1.0) == 0
        assert f.fake_memsets() == before + 1, k
    dev.set_atoms(box.XP, box.XP1, box.ITYP, box.STATU)
    dev.build_neighbors()
    for call in (dev.build_neighbors, lambda: dev.run(3, 1, 0, ctrl.H)):
        dev.build_neighbors()
        f.fake_refuse(b"k_scan_blocks")
        assert _hip_error(call)
        f.fake_refuse(b"")
        fills = f.fake_launches(b"k_fill_int")
        call()
        assert f.fake_launches(b"k_fill_int") == fills + 1
        call()
        assert f.fake_launches(b"k_fill_int") == fills + 1


@case
def pinned_ring(f):
    """Creating a context pins its own few words only, and works where no more can be pinned: copies
    are then plain ones.  So are those to the device, and those to the host of one part up to
    4 MB or of several between half a megabyte and four.  The first of the others pins the
    ring, which goes with the last context."""
    ring = 8 << 20
    for limit in (ring - 1, -1):
        f.fake_host_limit(limit)
        dev, boxes, _ = _device((30, 30, 30))      # 5.1 MB (2^20) of per-atom arrays
        other, _, _ = _device((26, 27, 29))        # 3.9
        other.get_atoms()
        dev.put_atoms(boxes[0].XP, None)
        few, _, _ = _device((12, 12, 14))          # 0.4
        few.get_forces()
        few.close()
        dev.set_atoms(boxes[0].XP, boxes[0].XP1, boxes[0].ITYP, boxes[0].STATU)
        small = f.fake_host_bytes()
        assert small < ring // 8
        have = small + (0 if limit > 0 else ring)
        for _ in range(2):
            # the runtime's memory holds 0x5a, and the kernels leave it
            assert all(set(a.tobytes()) == {0x5a} for a in dev.get_atoms())
            assert f.fake_host_bytes() == have
        tries = f.fake_host_allocs()
        dev.put_atoms(boxes[0].XP, boxes[0].XP1)
        x = dev.get_atoms()[0]      # the staging block as put_atoms left it: the velocities
        assert np.array_equal(x, boxes[0].XP1)
        assert f.fake_host_allocs() == tries        # refused once is refused while contexts live
        dev.close()
        assert f.fake_host_bytes() >= have - small
        other.close()
        assert f.fake_host_bytes() == 0
    few, _, _ = _device((12, 12, 14))
    small = f.fake_host_bytes()
    assert all(set(a.tobytes()) == {0x5a} for a in few.get_atoms())
    assert f.fake_host_bytes() == small + ring
    few.close()
    assert f.fake_host_bytes() == 0


@case
def pass_options(f):
    """The choice of the passes by size survives options set to what they are, and compaction switched
    on and off; MSM_PATH_BY_SIZE is reported for it and brings it back."""
    import msmpscu_amd._lib as L
    dev, _, _ = _device()
    opts = [L.MSM_OPT_FORCE_PATH, L.MSM_OPT_COMPACT_LIST, L.MSM_OPT_CHUNK_SWEEP, L.MSM_OPT_TABLE_LDS,
            L.MSM_OPT_LT_DENSITY_BLOCK, L.MSM_OPT_LT_DENSITY_WGS, L.MSM_OPT_LT_FORCE_BLOCK,
            L.MSM_OPT_LT_FORCE_WGS, L.MSM_OPT_FORCE_LANES]
    first = {o: dev.get_option(o) for o in opts}
    assert first[L.MSM_OPT_FORCE_PATH] == L.MSM_PATH_BY_SIZE == -1
    assert dev.pass_kernel() == "wide"
    for o in opts:
        dev.set_option(o, first[o])
        assert dev.pass_kernel() == "wide", o
    dev.set_option(L.MSM_OPT_COMPACT_LIST, 1)
    assert dev.pass_kernel() == "lds_table"
    dev.set_option(L.MSM_OPT_COMPACT_LIST, 0)
    assert dev.pass_kernel() == "wide"
    for o, v, kernel in ((L.MSM_OPT_FORCE_PATH, 2, "lds_table"), (L.MSM_OPT_TABLE_LDS, 0, "lanes"),
                         (L.MSM_OPT_LT_FORCE_BLOCK, 256, "lds_table"),
                         (L.MSM_OPT_FORCE_LANES, 1, "lds_table")):
        dev.set_option(o, v)
        assert dev.pass_kernel() == kernel and dev.get_option(o) == v
        assert dev.get_option(L.MSM_OPT_FORCE_PATH) == 2
        dev.set_option(L.MSM_OPT_FORCE_PATH, L.MSM_PATH_BY_SIZE)
        assert dev.pass_kernel() == "wide"
        assert {q: dev.get_option(q) for q in opts} == first
    assert L.lib().msm_set_option(dev.h, L.MSM_OPT_FORCE_PATH, -2) == 1      # MSM_ERR_ARG


@case
def table_lds_off(f):
    """MSM_OPT_TABLE_LDS 0 keeps the knots of the energy and stress passes out of LDS too."""
    import msmpscu_amd._lib as L
    dev, _, _ = _device((30, 30, 30))       # 54,000 atoms: knots in LDS by size
    dev.build_neighbors()

    def launches():     # k_*_w<..., lanes, TL>
        return [f.fake_launches(k) for k in (b"ELi1EEEvNS_8AtomsDevENS_7ListDevE", b"Li8ELi0EEEvNS_8AtomsDevENS_7ListDevE")]
    dev.calc_epot()
    dev.calc_atomic_stress()
    lds, glob = launches()
    assert lds == 3 and glob == 0       # energy; density and virial
    dev.set_option(L.MSM_OPT_TABLE_LDS, 0)
    dev.calc_epot()
    dev.calc_atomic_stress()
    assert launches() == [lds, 2]


@case
def autotune_fails(f):
    """An autotuner whose timing fails leaves every option as it was."""
    import msmpscu_amd._lib as L
    dev, _, _ = _device()
    dev.build_neighbors()
    opts = range(L.MSM_OPT_TRACK_DIS, L.MSM_OPT_CHUNK_SWEEP + 1)

    def state():
        return [dev.get_option(o) for o in opts]
    for setting in ((), ((L.MSM_OPT_FORCE_PATH, 4), (L.MSM_OPT_LT_FORCE_BLOCK, 512),
                         (L.MSM_OPT_BRICK_LANES, 4), (L.MSM_OPT_KERNEL_TIMING, 1)),
                    ((L.MSM_OPT_NLIST_KERNEL, 3), (L.MSM_OPT_COMPACT_LIST, 1))):
        for o, v in setting:
            dev.set_option(o, v)
        dev.build_neighbors()
        before = state()
        for k in (1, 3, 4, 5, 9, 15):       # the list kernels, then the passes
            f.fake_time_fail(k)
            assert _hip_error(lambda: dev.autotune(1))
            f.fake_time_fail(0)
            assert state() == before, k
            dev.build_neighbors()
    dev.autotune(1)


@case
def density_is_timed_once(f):
    """MSM_OPT_KERNEL_TIMING counts one density pass an evaluation of the loss and a quench step,
    whichever kernel makes it."""
    import msmpscu_amd._lib as L
    dev, boxes, ctrl = _device()
    dev.build_neighbors()
    n = boxes[0].NPRT
    ft, et, loss = np.zeros(3 * n), np.zeros(1), np.zeros(1)
    assert L.lib().msm_fm_set_targets(dev.h, L.dptr(ft), L.dptr(et), 1.0) == 0
    dev.set_option(L.MSM_OPT_KERNEL_TIMING, 1)
    for compact in (0, 1):
        dev.set_option(L.MSM_OPT_COMPACT_LIST, compact)
        dev.kernel_times()
        assert L.lib().msm_fm_loss_grad(dev.h, L.dptr(loss), None, 0, 0) == 0
        t = dev.kernel_times()
        assert (t["density"][1], t["force"][1]) == (1, 1), (compact, t)
        assert _hip_error(lambda: dev.dyn_damp(1, 0.0, ctrl.H))      # (no kernel leaves the note)
        t = dev.kernel_times()
        assert (t["density"][1], t["force"][1]) == (1, 1), (compact, t)


@case
def copy_out_in_little_memory(f):
    """All arrays at once leave through one block of 100 bytes an atom; where that cannot be had, one
    after another through 24."""
    import msmpscu_amd._lib as L
    dev, boxes, _ = _device((16, 16, 17))
    n = boxes[0].NPRT
    f.fake_dev_limit(24 * n)
    for _ in range(2):
        assert all(set(a.tobytes()) == {0x5a} for a in dev.get_atoms())
    dev.close()
    dev, boxes, _ = (f.fake_dev_limit(-1), _device((16, 16, 17)))[1]
    f.fake_dev_limit(24 * n - 1)
    try:
        dev.get_atoms()
        raise AssertionError("copied through nothing")
    except L.MSMError as e:
        assert e.code == 3      # MSM_ERR_NOMEM
    dev.close()


@case
def refused_in_the_middle(f):
    """A rebuild whose sort is refused leaves the atoms where they are (the runtime's memory is what it
    was: nothing moved to the other buffers) and no list; a pass that is refused is no candidate of the
    autotuner, and no error while others run; a list kernel that is, is one."""
    import msmpscu_amd._lib as L
    dev, boxes, ctrl = _device()
    dev.build_neighbors()
    for kernel in (b"k_sort_small", b"k_order_move", b"k_nlist"):
        f.fake_refuse(kernel)
        lists = f.fake_launches(b"k_nlist")
        assert _hip_error(dev.build_neighbors)
        assert f.fake_launches(b"k_nlist") == lists
        f.fake_refuse(b"")
        try:
            dev.calc_force()
            raise AssertionError("forces from no list")
        except L.MSMError as e:
            assert e.code == 7      # MSM_ERR_STATE
        dev.build_neighbors()

    def state():
        return [dev.get_option(o) for o in range(L.MSM_OPT_TRACK_DIS, L.MSM_OPT_CHUNK_SWEEP + 1)]
    before = state()
    for kernel in (b"k_nlist_small", b"k_order_move", b"k_d"):
        f.fake_refuse(kernel)
        assert _hip_error(lambda: dev.autotune(1)), kernel
        assert state() == before
        f.fake_refuse(b"")
        dev.build_neighbors()
    f.fake_refuse(b"k_force_w")
    assert dev.autotune(1)["force_path"] not in (L.MSM_PATH_BY_SIZE, 1, 2, 4)
    dev.calc_force()


@pytest.mark.parametrize("name", sorted(CASES))
def test_host_path(fake, name):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), name, fake],
                       cwd=os.path.dirname(HERE), stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stdout


if __name__ == "__main__":
    import ctypes
    runtime = ctypes.CDLL(sys.argv[2], mode=ctypes.RTLD_GLOBAL)
    for fn in ("fake_host_bytes", "fake_host_allocs", "fake_dev_bytes", "fake_memsets"):
        getattr(runtime, fn).restype = ctypes.c_long
    for fn in ("fake_host_limit", "fake_dev_limit"):
        getattr(runtime, fn).argtypes = [ctypes.c_long]
        getattr(runtime, fn).restype = None
    sys.path.insert(0, os.path.dirname(HERE))
    CASES[sys.argv[1]](runtime)
    print("ok")
