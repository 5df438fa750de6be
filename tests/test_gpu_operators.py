"""GPU parity tests of the HIP operators and solvers against the FP64 oracle.

Tolerances (FP32 device vs FP64 oracle): forward / transpose outputs within
1e-5 relative L2; adjoint identity <Ax, y> = <x, A'y> within 1e-6 relative;
reconstructions within 1e-3 relative L2 at equal iterations.
"""
import numpy as np
import pytest

import oracle as O
from helpers import geometry_tt, random_sir, random_tt, rel_l2, rng

pytestmark = pytest.mark.gpu

TOL_OP = 1e-5
TOL_ADJ = 1e-6
TOL_REC = 1e-3


@pytest.fixture(scope="module", autouse=True)
def _gpu(require_gpu):
    import mbrec
    mbrec.lib()
    yield


def _log(msg):
    print(msg, flush=True)


# --- MEX drop-ins (host FP64 in/out) -------------------------------------------------
@pytest.mark.parametrize("W,P,D,nT,R,spill", [(1, 1000, 16, 300, 2.6666666666666665, 0.0),
                                              (3, 777, 9, 257, 3.3333333333333335, 0.15),
                                              (2, 64, 5, 128, 1.6, 0.3),
                                              (1, 130, 4, 96, 2.0, 0.2)])
def test_mex_das_matches_oracle(W, P, D, nT, R, spill):
    from mbrec.mex import forwardDelayAndSumMex, transposeDelayAndSumMex
    _log(f"mex_das W={W} P={P} D={D} nT={nT} R={R}")
    tt = random_tt(P, D, nT, R, seed=P + D, spill=spill)
    x = rng(1).uniform(0, 1, (W, P))
    y = forwardDelayAndSumMex(x, tt, np.int32(nT), R)
    yo = O.forward_das(x, tt, nT, R)
    assert y.shape == (W, nT, D)
    assert rel_l2(y, yo) < TOL_OP
    s = rng(2).standard_normal((W, nT, D))
    xt = transposeDelayAndSumMex(s, tt, R)
    assert xt.shape == (W, P)
    assert rel_l2(xt, O.transpose_das(s, tt, R)) < TOL_OP


@pytest.mark.parametrize("W", [1, 3])
def test_mex_das_on_an_arc_geometry(W):
    """The DAS drop-ins with the travel times of a real grid (96 x 80 pixels, 40 detectors of
    the arc): the MEX path reads the column length off the table and runs the 2-D tile
    kernels; results against the oracle's loops."""
    from mbrec.mex import forwardDelayAndSumMex, transposeDelayAndSumMex
    _log(f"mex_das on an arc geometry W={W}")
    m = _geometry_model(96, 80, 40, 700, 1e-4, sir=False, sigma=1.0)
    orc = _oracle_of(m)
    tt = np.asfortranarray(orc.tt.T)   # [P x D]
    D, nT = m.shape_sinogram
    x = rng(41).uniform(0, 1, (W, tt.shape[0]))
    y = forwardDelayAndSumMex(x, tt, np.int32(nT), orc.R)
    assert rel_l2(y, O.forward_das(x, tt, nT, orc.R)) < TOL_OP
    sg = rng(42).standard_normal((W, nT, D))
    xt = transposeDelayAndSumMex(sg, tt, orc.R)
    assert rel_l2(xt, O.transpose_das(sg, tt, orc.R)) < TOL_OP


@pytest.mark.parametrize("W,P,D,nT,R,Ls", [(1, 500, 8, 200, 2.6666666666666665, 9),
                                           (2, 333, 6, 150, 1.6, 15),
                                           (5, 70, 3, 90, 3.3333333333333335, 4)])
def test_mex_sir_matches_oracle(W, P, D, nT, R, Ls):
    from mbrec.mex import forwardMex, transposeMex
    _log(f"mex_sir W={W} P={P} D={D} nT={nT} R={R} Ls={Ls}")
    tt = random_tt(P, D, nT, R, seed=7, spill=0.1)
    sidx, sir, se = random_sir(P, D, Ls=Ls, Nsir=11, seed=8)
    x = rng(3).uniform(0, 1, (W, P))
    y = forwardMex(x, sidx, tt, sir, np.int32(nT), se, R)
    assert rel_l2(y, O.forward_sir(x, sidx, tt, sir, nT, se, R)) < TOL_OP
    s = rng(4).standard_normal((W, nT, D))
    xt = transposeMex(s, sidx, tt, sir, se, R)
    assert rel_l2(xt, O.transpose_sir(s, sidx, tt, sir, se, R)) < TOL_OP


def test_mex_known_answers():
    from mbrec.mex import forwardDelayAndSumMex, forwardMex
    y = forwardDelayAndSumMex(np.array([[2.0]]), np.array([[10.25]]), np.int32(20), 2.5)
    want = np.zeros(20); want[8:13] = [0.2, 1.0, 1.8, 1.4, 0.6]
    np.testing.assert_allclose(y[0, :, 0], want, atol=1e-6)
    sir = np.array([[0.0, 1.0, 2.0, 3.0, 0.0]]).T
    y = forwardMex(np.array([[1.0]]), np.array([[1]], dtype=np.int32), np.array([[10.0]]), sir, np.int32(16),
                   np.array([[2], [4]], dtype=np.int32), 1.5)
    want = np.zeros(16); want[8:13] = [1 / 3, 5 / 3, 10 / 3, 11 / 3, 1.0]
    np.testing.assert_allclose(y[0, :, 0], want, atol=1e-6)


# --- device plans (tiled pixel order) ------------------------------------------------
def _plan_problem(Nz, Nx, D, nT, R, seed, sir=False):
    import torch
    from mbrec.model import DevicePlan
    P = Nz * Nx
    tt = random_tt(P, D, nT, R, seed=seed, spill=0.05)
    kw = {}
    if sir:
        sidx, s, se = random_sir(P, D, Ls=13, Nsir=9, seed=seed + 1)
        kw["sir"] = (sidx.T, s.T, se.T)
    plan = DevicePlan(Nz, Nx, D, nT, R, tt.T, **kw)
    return plan, tt, kw, torch


@pytest.mark.parametrize("sir", [False, True])
@pytest.mark.parametrize("B", [1, 3, 6, 20, 64])
def test_device_mex_ops_batched(sir, B):
    Nz, Nx, D, nT, R = 37, 29, 12, 220, 2.6666666666666665
    _log(f"device_mex sir={sir} B={B}")
    plan, tt, kw, torch = _plan_problem(Nz, Nx, D, nT, R, seed=20 + B, sir=sir)
    x = rng(5).uniform(0, 1, (B, Nx, Nz))
    y = plan.forward(torch.tensor(x, dtype=torch.float32).cuda(), model=False).cpu().numpy()
    xo = x.reshape(B, -1)
    if sir:
        sidx, s, se = (a.T for a in kw["sir"])
        yo = O.forward_sir(xo, sidx, tt, s, nT, se, R)
    else:
        yo = O.forward_das(xo, tt, nT, R)
    yo = np.transpose(yo, (0, 2, 1))          # [W x nT x D] -> (W, D, nT)
    assert rel_l2(y, yo) < TOL_OP
    sg = rng(6).standard_normal((B, D, nT))
    xt = plan.transpose(torch.tensor(sg, dtype=torch.float32).cuda(), model=False).cpu().numpy()
    sgm = np.transpose(sg, (0, 2, 1))
    xto = O.transpose_sir(sgm, sidx, tt, s, se, R) if sir else O.transpose_das(sgm, tt, R)
    assert rel_l2(xt.reshape(B, -1), xto) < TOL_OP


def test_set_sir_twice_replaces_tables():
    """A second mbrec_plan_set_sir with longer windows, more SIR entries and a different
    table length replaces every SIR-dependent table and the workspace sized from them:
    the batch (band form) and one-sinogram forwards and the transposes match the oracle of
    the new tables."""
    import torch
    from mbrec.model import DevicePlan
    Nz, Nx, D, nT, R = 33, 31, 10, 240, 2.6666666666666665
    P = Nz * Nx
    tt = random_tt(P, D, nT, R, seed=41, spill=0.05)
    first = random_sir(P, D, Ls=7, Nsir=5, seed=42)
    second = random_sir(P, D, Ls=29, Nsir=13, seed=43)
    plan = DevicePlan(Nz, Nx, D, nT, R, tt.T, sir=tuple(a.T for a in first))
    for B in (1, 20):           # build the workspace (and band rows) for the first tables
        plan.forward(torch.rand((B, P), device="cuda"), model=False)
    plan.set_sir(*(a.T for a in second))
    sidx, s, se = second
    for B in (1, 20):
        _log(f"set_sir twice B={B}")
        x = rng(44 + B).uniform(0, 1, (B, P))
        y = plan.forward(torch.tensor(x, dtype=torch.float32).cuda(), model=False).cpu().numpy()
        yo = np.transpose(O.forward_sir(x, sidx, tt, s, nT, se, R), (0, 2, 1))
        assert rel_l2(y, yo) < TOL_OP
        sg = rng(45 + B).standard_normal((B, D, nT))
        xt = plan.transpose(torch.tensor(sg, dtype=torch.float32).cuda(), model=False).cpu().numpy()
        xto = O.transpose_sir(np.transpose(sg, (0, 2, 1)), sidx, tt, s, se, R)
        assert rel_l2(xt.reshape(B, -1), xto) < TOL_OP
    plan.close()


def test_one_sinogram_forward_larger_image():
    """The one-sinogram pull (image gathered into device slot order, slot-indexed records)
    on a 208 x 208 image of 169 device tiles gives the oracle's forward."""
    Nz, Nx, D, nT, R = 208, 208, 12, 220, 2.6666666666666665
    _log("one-sinogram forward 208x208")
    plan, tt, kw, torch = _plan_problem(Nz, Nx, D, nT, R, seed=77)
    x = rng(7).uniform(0, 1, (1, Nx, Nz))
    y = plan.forward(torch.tensor(x, dtype=torch.float32).cuda(), model=False).cpu().numpy()
    yo = np.transpose(O.forward_das(x.reshape(1, -1), tt, nT, R), (0, 2, 1))
    assert rel_l2(y, yo) < TOL_OP


@pytest.mark.parametrize("sir", [False, True])
@pytest.mark.parametrize("B", [1, 8, 20, 32, 64])
def test_every_launch_variant_matches_oracle(sir, B):
    """Each gather variant and scatter choice valid for B gives the oracle's result."""
    from mbrec import _lib
    Nz, Nx, D, nT, R = 24, 20, 10, 200, 2.6666666666666665
    _log(f"launch variants sir={sir} B={B}")
    plan, tt, kw, torch = _plan_problem(Nz, Nx, D, nT, R, seed=40 + B, sir=sir)
    x = rng(15).uniform(0, 1, (B, Nx, Nz))
    sg = rng(16).standard_normal((B, D, nT))
    xo = x.reshape(B, -1)
    sgm = np.transpose(sg, (0, 2, 1))
    if sir:
        sidx, s, se = (a.T for a in kw["sir"])
        yo = np.transpose(O.forward_sir(xo, sidx, tt, s, nT, se, R), (0, 2, 1))
        xto = O.transpose_sir(sgm, sidx, tt, s, se, R)
    else:
        yo = np.transpose(O.forward_das(xo, tt, nT, R), (0, 2, 1))
        xto = O.transpose_das(sgm, tt, R)
    xd = torch.tensor(x, dtype=torch.float32).cuda()
    sd = torch.tensor(sg, dtype=torch.float32).cuda()
    n_ok = 0
    for gv in range(_lib.lib().mbrec_num_gather_variants()):
        for sc in (1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 16, -16, -32, -64, -116, -164, -216, -264, -364, -464,
                   -564, -664, -764, -864, -964, -1064, -1164, 1000, 1001, 1002, 1003, 1004):
            try:
                plan.set_launch(B, gv, sc)
            except Exception:
                continue
            n_ok += 1
            y = plan.forward(xd, model=False).cpu().numpy()
            xt = plan.transpose(sd, model=False).cpu().numpy()
            assert rel_l2(y, yo) < TOL_OP, (gv, sc)
            assert rel_l2(xt.reshape(B, -1), xto) < TOL_OP, (gv, sc)
    assert n_ok >= 1
    plan.set_launch(B, -1, 0)


@pytest.mark.parametrize("length,B", [(1, 1), (24, 1), (25, 1), (31, 1), (32, 1), (24, 2), (25, 33), (31, 32), (32, 4),
                                      (8, 64), (24, 67), (30, 33), (31, 33)])
def test_sir_forward_band_edges(length, B):
    """The band forms of the SIR forward at the window lengths where they change (24: bands that
    slide, 31: longest window of a band, 32: the forms without bands) and at the edges of a
    wave's sinograms; random travel times put taps on both ends of the sample axis, every
    record list is odd-sized or empty somewhere, and 67 detectors leave workgroups partly idle."""
    import torch
    from mbrec.model import DevicePlan
    Nz, Nx, D, nT, R, Ls = 11, 13, 67, 150, 2.6666666666666665, 35
    _log(f"sir band edges length={length} B={B}")
    g = rng(500 + length)
    tt = random_tt(Nz * Nx, D, nT, R, 7, margin=-6)
    nsir = 9
    sir = g.standard_normal((Ls, nsir))
    se = np.zeros((2, nsir), dtype=np.int32)
    for k in range(nsir):
        n = length if k == 0 else int(g.integers(1, length + 1))
        s0 = int(g.integers(1, Ls - n + 2))
        se[:, k] = (s0, s0 + n - 1)
    se[:, nsir - 1] = (3, 2)          # no taps
    sidx = g.integers(1, nsir + 1, size=(Nz * Nx, D)).astype(np.int32)
    plan = DevicePlan(Nz, Nx, D, nT, R, np.ascontiguousarray(tt.T),
                      sir=(np.ascontiguousarray(sidx.T), np.ascontiguousarray(sir.T), np.ascontiguousarray(se.T)))
    x = g.uniform(0, 1, (B, Nx, Nz))
    yo = np.transpose(O.forward_sir(x.reshape(B, -1), sidx, tt, sir, nT, se, R), (0, 2, 1))
    y = plan.forward(torch.tensor(x, dtype=torch.float32).cuda(), model=False).cpu().numpy()
    assert rel_l2(y, yo) < TOL_OP
    assert np.abs(y - yo).max() < 1e-4 * np.abs(yo).max()
    if B == 1:
        return
    # the band form is there up to 31 taps, up to 30 above 32 sinograms, and whatever the workspace held before
    has_band = length < (31 if B > 32 else 32)
    for _ in range(2):
        if has_band:
            plan.set_launch(B, -1, 1004)
            assert np.array_equal(plan.forward(torch.tensor(x, dtype=torch.float32).cuda(), model=False).cpu().numpy(), y)
        else:
            with pytest.raises(Exception):
                plan.set_launch(B, -1, 1004)
        plan.set_launch(B, -1, 0)
        plan.forward(torch.zeros((70, Nx, Nz), device="cuda"), model=False)


@pytest.mark.parametrize("B", [2, 4, 13, 16, 17, 28, 33, 70])
@pytest.mark.parametrize("crop", ["inside", "start", "end"])
def test_sir_transpose_groups_match_oracle(B, crop):
    """The matrix-core SIR transpose on an arc geometry (grid ending inside tiles, batches around
    16 and 32 columns), with every tap on the sample axis and with travel times that leave it at
    its start or end, where the groups' windows are moved back and taps drop out; empty
    windows among the SIR entries."""
    import torch
    from mbrec.model import DevicePlan
    Nz, Nx, D, R, Ls = 37, 53, 9, 2.6666666666666665, 31
    _log(f"sir groups B={B} crop={crop}")
    tt = geometry_tt(Nz, Nx, 1e-4, D, 0.01, 160.0, 1500.0, 4e7).reshape(D, -1)
    lo, hi = int(tt.min()), int(tt.max()) + 1
    nT = hi - lo + 60
    tt = tt - lo + {"inside": 30, "start": -50, "end": 130}[crop]
    g = rng(900)
    nsir = 40
    sir = g.standard_normal((Ls, nsir))
    se = np.zeros((2, nsir), dtype=np.int32)
    for k in range(nsir):
        n = int(g.integers(14, 25))
        s0 = int(g.integers(3, 6))
        se[:, k] = (s0, s0 + n - 1)
    se[:, 0] = (3, 2)
    sidx = g.integers(1, nsir + 1, size=(Nz * Nx, D)).astype(np.int32)
    plan = DevicePlan(Nz, Nx, D, nT, R, tt, sir=(np.ascontiguousarray(sidx.T), np.ascontiguousarray(sir.T),
                                                 np.ascontiguousarray(se.T)))
    sg = g.standard_normal((B, D, nT))
    xto = O.transpose_sir(np.transpose(sg, (0, 2, 1)), sidx, np.ascontiguousarray(tt.T), sir, se, R)
    sd = torch.tensor(sg, dtype=torch.float32).cuda()
    ran = 0
    for v in (-1, 59, 60, 61, 62):
        try:
            plan.set_launch(B, v, 0)
        except Exception:
            continue
        ran += v > 0
        xt = plan.transpose(sd, model=False).cpu().numpy()
        assert rel_l2(xt.reshape(B, -1), xto) < TOL_OP, v
    assert ran == 4      # the geometry's pairs fit the groups


def test_sir_group_tables_follow_the_sir_tables():
    """The tables of the matrix-core SIR transpose go with SIR windows too long for them (36 taps; the older forms
    run) and come back with the first ones, and the transpose that allocates nothing finds them there."""
    import torch
    from mbrec import _lib
    _log("SIR group tables")
    D, nT, Nz, Nx = 12, 300, 40, 44
    m = _geometry_model(Nz, Nx, D, nT, 1e-4, sir=True, sigma=1.0)
    d, plan = m.Data, m.plan
    tt, R = _oracle_of(m).tt.T, _oracle_of(m).R
    first = (d.SPMRIndices.reshape(D, -1), d.SPMR, d.SPMRTimestepIndexStartAndEnd)
    g = rng(39)
    long_ = (g.integers(1, 6, size=(D, Nz * Nx)).astype(np.int32), g.standard_normal((5, 61)),
             np.tile(np.array([[12, 47]], dtype=np.int32), (5, 1)))
    sg = g.standard_normal((4, D, nT))
    sd = torch.tensor(sg, dtype=torch.float32).cuda()
    seen = []
    for sidx, table, se in (first, long_, first):
        plan.set_sir(sidx, table, se)
        if se is long_[2]:
            with pytest.raises(Exception):
                plan.set_launch(4, 61, 0)
        else:
            got = torch.full((4, Nz * Nx), float("nan"), device="cuda")
            _lib.check(_lib.lib().mbrec_model_transpose_noalloc_dev(plan.h, sd.data_ptr(), got.data_ptr(), 4,
                                                                    _lib.stream_handle()))
            assert torch.equal(got, plan.transpose(sd).reshape(4, -1))
            plan.set_launch(4, 61, 0)
        ref = O.transpose_sir(np.transpose(sg, (0, 2, 1)), sidx.T, tt, table.T, se.T, R)
        seen.append(plan.transpose(sd, model=False).cpu().numpy().reshape(4, -1))
        assert rel_l2(seen[-1], ref) < TOL_OP
    assert np.array_equal(seen[0], seen[2])
    assert 0 < plan.device_bytes < 1 << 40


@pytest.mark.parametrize("sir", [False, True])
@pytest.mark.parametrize("B", [4, 9, 16, 28, 64])
def test_transpose_keeps_non_finite_samples_apart(sir, B):
    """Infinite and NaN samples reach the pixels of their own pairs' taps only, and their own sinogram only:
    every batch gather against the record-lane form (2), which reads a pair's own bins and no others.  The
    SIR windows hold zeros, whose taps count."""
    import torch
    from mbrec.model import DevicePlan
    _log(f"non-finite samples sir={sir} B={B}")
    Nz, Nx, D, R, Ls = 37, 53, 9, 2.6666666666666665, 31
    tt = geometry_tt(Nz, Nx, 1e-4, D, 0.01, 160.0, 1500.0, 4e7).reshape(D, -1)
    tt = tt - int(tt.min()) + 10                       # some taps before the first sample
    nT = int(tt.max()) + 5
    g = rng(901)
    kw = {}
    if sir:
        nsir = 40
        sir_t = g.standard_normal((nsir, Ls))
        se = np.zeros((nsir, 2), dtype=np.int32)
        for k in range(nsir):
            s0 = int(g.integers(3, 6))
            se[k] = (s0, s0 + int(g.integers(14, 25)) - 1)
            sir_t[k, s0 + 4] = 0.0
            sir_t[k, s0 + 6] = -0.0
        kw["sir"] = (g.integers(1, nsir + 1, size=(D, Nz * Nx)).astype(np.int32), sir_t, se)
    plan = DevicePlan(Nz, Nx, D, nT, R, tt, **kw)
    y = g.standard_normal((B, D, nT)).astype(np.float32)
    for b, d, t, v in [(0, 4, nT // 2, np.inf), (1, 2, nT // 3, -np.inf), (3, 7, 2, np.nan), (B - 1, 8, nT - 3, np.inf),
                       (B - 1, 1, nT // 4, np.nan)]:
        y[b, d, t] = v
    yd = torch.tensor(y).cuda()
    plan.set_launch(B, 2, 0)
    want = plan.transpose(yd, model=False).cpu().numpy()
    bad = ~np.isfinite(want)
    assert bad[[0, 1, B - 1]].any(axis=(1, 2)).all() and not bad[2].any() and bad.mean() < 0.6
    ran = []
    for v in range(-1, 63):
        try:
            plan.set_launch(B, v, 0)
        except Exception:
            continue
        ran.append(v)
        x = plan.transpose(yd, model=False).cpu().numpy()
        assert np.array_equal(~np.isfinite(x), bad), v
        assert rel_l2(x[~bad], want[~bad]) < TOL_OP, v
    assert not sir or {59, 60, 61, 62}.issubset(ran)
    assert sir or B < 9 or {55, 56, 57, 58}.issubset(ran)


def test_default_forward_choice_can_be_set():
    """The automatic forward choice of batches of 9 to 12 is one that set_launch and the autotuner take."""
    _log("default forward choice")
    plan, _, _, _ = _plan_problem(13, 11, 24, 150, 2.6666666666666665, seed=92)
    for B in (9, 10, 12, 13):
        plan.set_launch(B, -1, -864)
    for B in (1, 8):
        with pytest.raises(Exception):
            plan.set_launch(B, -1, -864)


@pytest.mark.parametrize("sir", [False, True])
@pytest.mark.parametrize("B", [1, 12, 64])
def test_autotuned_launch_matches_oracle(sir, B):
    """The autotuner (ramp-up, first pass, refinement of the three fastest) returns a valid
    launch choice for B, and the operators under it give the oracle's result."""
    Nz, Nx, D, nT, R = 24, 20, 10, 200, 2.6666666666666665
    _log(f"autotune sir={sir} B={B}")
    plan, tt, kw, torch = _plan_problem(Nz, Nx, D, nT, R, seed=60 + B, sir=sir)
    gv, sc = plan.autotune(B, 2)
    plan.set_launch(B, gv, sc)   # raises if the choice is not valid for B
    x = rng(17).uniform(0, 1, (B, Nx, Nz))
    sg = rng(18).standard_normal((B, D, nT))
    xo, sgm = x.reshape(B, -1), np.transpose(sg, (0, 2, 1))
    if sir:
        sidx, s, se = (a.T for a in kw["sir"])
        yo = np.transpose(O.forward_sir(xo, sidx, tt, s, nT, se, R), (0, 2, 1))
        xto = O.transpose_sir(sgm, sidx, tt, s, se, R)
    else:
        yo = np.transpose(O.forward_das(xo, tt, nT, R), (0, 2, 1))
        xto = O.transpose_das(sgm, tt, R)
    y = plan.forward(torch.tensor(x, dtype=torch.float32).cuda(), model=False).cpu().numpy()
    xt = plan.transpose(torch.tensor(sg, dtype=torch.float32).cuda(), model=False).cpu().numpy()
    assert rel_l2(y, yo) < TOL_OP, (gv, sc)
    assert rel_l2(xt.reshape(B, -1), xto) < TOL_OP, (gv, sc)


@pytest.mark.parametrize("B", [9, 12, 13, 16, 17, 28, 32, 33, 48, 64, 65, 70])
@pytest.mark.parametrize("smooth", [True, False])
def test_default_batch_forms_match_oracle(B, smooth):
    """The automatic forward and gather of a plan without SIR around the batch sizes where they
    change (12, 16, 32, 64; several workgroups' columns), on an arc geometry whose tile windows
    fit the LDS gather (its grid ends inside a tile in both directions) and on random travel
    times, where the forms without windows run."""
    import torch
    _log(f"default batch forms B={B} smooth={smooth}")
    if smooth:
        m = _geometry_model(57, 70, 24, 700, 1e-4, sir=False, sigma=1.0)
        plan, tt, R, shape = m.plan, _oracle_of(m).tt.T, _oracle_of(m).R, (70, 57)
        D, nT = m.shape_sinogram
    else:
        D, nT, R, shape = 12, 160, 2.6666666666666665, (20, 23)
        plan, tt, _, _ = _plan_problem(23, 20, D, nT, R, seed=70 + B)
    x = rng(33).uniform(0, 1, (B, *shape))
    sg = rng(34).standard_normal((B, D, nT))
    yo = np.transpose(O.forward_das(x.reshape(B, -1), tt, nT, R), (0, 2, 1))
    xto = O.transpose_das(np.transpose(sg, (0, 2, 1)), tt, R)
    y = plan.forward(torch.tensor(x, dtype=torch.float32).cuda(), model=False).cpu().numpy()
    xt = plan.transpose(torch.tensor(sg, dtype=torch.float32).cuda(), model=False).cpu().numpy()
    assert rel_l2(y, yo) < TOL_OP
    assert rel_l2(xt.reshape(B, -1), xto) < TOL_OP


@pytest.mark.parametrize("B", [12, 13, 28, 33, 64, 70])
def test_forward_keeps_non_finite_pixels_apart(B):
    """Infinite and NaN pixels reach the samples of their own pairs only, and their own sinogram only:
    every batch form against the form with a thread per bin (forward choice 1), which reads the
    records of its bin and no others."""
    import torch
    _log(f"non-finite pixels B={B}")
    Nz, Nx, D, nT = 13, 11, 24, 150
    plan, tt, _, _ = _plan_problem(Nz, Nx, D, nT, 2.6666666666666665, seed=90)
    x = rng(91).uniform(0, 1, (B, Nx, Nz)).astype(np.float32)
    for k, (b, v) in enumerate([(0, np.inf), (1, -np.inf), (5, np.nan), (B - 1, np.inf), (B - 1, np.nan)]):
        x[b, 3 + k, 4] = v
    xd = torch.tensor(x).cuda()
    plan.set_launch(B, -1, 1)
    want = plan.forward(xd, model=False).cpu().numpy()
    bad = ~np.isfinite(want)
    assert bad[[0, 1, 5, B - 1]].any(axis=(1, 2)).all() and not bad[[2, 3, 4]].any() and bad.mean() < 0.05
    ran = 0
    for c in [0] + [-lb - 100 * mode for mode in range(12) for lb in (16, 32, 64)]:
        try:
            plan.set_launch(B, -1, c)
        except Exception:
            continue
        ran += c < 0
        y = plan.forward(xd, model=False).cpu().numpy()
        assert np.array_equal(~np.isfinite(y), bad), c
        assert rel_l2(y[~bad], want[~bad]) < TOL_OP, c
    assert ran >= 9


@pytest.mark.parametrize("B", [13, 28, 64])
def test_batch_gather_sums_as_close_as_compensated(B):
    """The LDS gathers of batches without SIR (55 to 58) add up 256 detectors of one sign: their distance to
    the FP64 oracle is no larger than that of the compensated forms (2: record lanes, 7: batch lanes);
    what those share, the 32-bit interpolation weights, allows 1 % between them."""
    import torch
    _log(f"gather sums B={B}")
    m = _geometry_model(57, 70, 256, 700, 1e-4, sir=False, sigma=1.0)
    tt, R = _oracle_of(m).tt.T, _oracle_of(m).R
    sg = 0.5 + rng(36).uniform(0, 1, (B, 256, 700))
    ref = O.transpose_das(np.transpose(sg, (0, 2, 1)), tt, R)
    sd = torch.tensor(sg, dtype=torch.float32).cuda()
    err = {}
    for v in (2, 7, 55, 56, 57, 58):
        m.plan.set_launch(B, v, 0)
        err[v] = rel_l2(m.plan.transpose(sd, model=False).cpu().numpy().reshape(B, -1), ref)
    print(B, {k: f"{e:.3e}" for k, e in err.items()}, flush=True)
    assert max(err[v] for v in (55, 56, 57, 58)) <= 1.01 * min(err[2], err[7])


@pytest.mark.parametrize("B,v", [(4, 61), (8, 61), (16, 61), (17, 59), (28, 59), (64, 59)])
def test_sir_batch_gather_sums_as_close_as_before(B, v):
    """The matrix-core SIR transpose adds up 75 detectors of one sign: its distance to the FP64 oracle is no
    larger than that of the form it replaces for the batch, compensated record lanes (2) up to 16
    sinograms, the vector tile form (39) above; 1 % for what those share."""
    import torch
    _log(f"SIR gather sums B={B}")
    m = _geometry_model(37, 40, 75, 700, 1e-4, sir=True, sigma=1.0)
    tt, d = _oracle_of(m).tt.T, m.Data
    sg = 0.5 + rng(37).uniform(0, 1, (B, 75, 700))
    ref = O.transpose_sir(np.transpose(sg, (0, 2, 1)), d.SPMRIndices.reshape(75, -1).T, tt, d.SPMR.T,
                          d.SPMRTimestepIndexStartAndEnd.T, _oracle_of(m).R)
    sd = torch.tensor(sg, dtype=torch.float32).cuda()
    err = {}
    for k in (-1, v, 2 if B <= 16 else 39):
        m.plan.set_launch(B, k, 0)
        err[k] = rel_l2(m.plan.transpose(sd, model=False).cpu().numpy().reshape(B, -1), ref)
    print(B, {k: f"{e:.3e}" for k, e in err.items()}, flush=True)
    assert err[-1] == err[v] <= 1.01 * err[2 if B <= 16 else 39]


@pytest.mark.parametrize("B", [2, 28, 64])
def test_sir_forward_sums_as_close_as_before(B):
    """The matrix-core SIR forward adds up 200 x 200 pixels of one sign: its distance to the FP64 oracle is no
    larger than that of the vector pull form (1000), which sums a sample's records one by one as the form
    before it did."""
    import torch
    _log(f"SIR forward sums B={B}")
    D, nT, n = 6, 1000, 200
    m = _geometry_model(n, n, D, nT, 1e-4, sir=True, sigma=1.0)
    tt, d = _oracle_of(m).tt.T, m.Data
    g = rng(38)
    c, r2 = g.uniform(0, n, (2, B, 1, 1)), ((np.arange(n)[:, None], np.arange(n)[None, :]))
    x = (0.5 + g.uniform(0, 1, (B, 1, 1)) * ((r2[0] - c[0]) ** 2 + (r2[1] - c[1]) ** 2 < 50.0 ** 2)).astype(np.float32)
    ref = np.transpose(O.forward_sir(x.reshape(B, -1), d.SPMRIndices.reshape(D, -1).T, tt, d.SPMR.T, nT,
                                     d.SPMRTimestepIndexStartAndEnd.T, _oracle_of(m).R), (0, 2, 1))
    xd = torch.tensor(x, dtype=torch.float32).cuda()
    err = {}
    for k in (0, 1004, 1000):
        m.plan.set_launch(B, -1, k)
        err[k] = rel_l2(m.plan.forward(xd, model=False).cpu().numpy(), ref)
    print(B, {k: f"{e:.3e}" for k, e in err.items()}, flush=True)
    assert err[0] == err[1004] <= err[1000]


@pytest.mark.parametrize("B", [13, 16, 28, 33, 64])
def test_lds_gather_many_detectors_match_oracle(B):
    """The LDS gathers of batches without SIR with more than eight detectors in a group and a last group that
    is shorter (75 detectors in groups of 38 and 19): all four forms are valid on this geometry, one of them is
    the automatic choice."""
    import torch
    _log(f"LDS gather 75 detectors B={B}")
    m = _geometry_model(57, 70, 75, 700, 1e-4, sir=False, sigma=1.0)
    tt, R = _oracle_of(m).tt.T, _oracle_of(m).R
    sg = rng(34).standard_normal((B, 75, 700))
    ref = O.transpose_das(np.transpose(sg, (0, 2, 1)), tt, R)
    sd = torch.tensor(sg, dtype=torch.float32).cuda()
    out = {}
    for v in (55, 56, 57, 58, -1):
        m.plan.set_launch(B, v, 0)
        out[v] = m.plan.transpose(sd, model=False).cpu().numpy().reshape(B, -1)
        assert rel_l2(out[v], ref) < TOL_OP, v
    assert any(np.array_equal(out[-1], out[v]) for v in (55, 56, 57, 58))


@pytest.mark.parametrize("B", [4, 16, 17, 33])
@pytest.mark.parametrize("h,rows", [(1e-4, 256), (6e-5, 192), (2e-5, 128)])
def test_sir_transpose_groups_many_detectors(h, rows, B):
    """The matrix-core SIR transpose with more than eight detectors in a group and a shorter last group (75
    detectors in groups of 19 and 10), for the three sizes of its row buffer (the samples that a tile's pairs
    span, three rows each, in steps of 64 rows)."""
    import torch
    from mbrec.model import DevicePlan
    Nz, Nx, D, R, Ls = 37, 53, 75, 2.6666666666666665, 31
    _log(f"SIR groups 75 detectors B={B} h={h}")
    tt = geometry_tt(Nz, Nx, h, D, 0.01, 160.0, 1500.0, 4e7).reshape(D, -1)
    tt = tt - int(tt.min()) + 30
    nT = int(tt.max()) + 60
    g = rng(902)
    nsir = 40
    se = np.zeros((nsir, 2), dtype=np.int32)
    for k in range(nsir):
        se[k, 0] = g.integers(3, 6)
        se[k, 1] = se[k, 0] + g.integers(14, 25) - 1
    sir = g.standard_normal((nsir, Ls))
    sidx = g.integers(1, nsir + 1, size=(D, Nz * Nx)).astype(np.int32)
    first = np.floor(tt).astype(int).reshape(D, Nx, Nz) + se[sidx - 1, 0].reshape(D, Nx, Nz)
    last = np.floor(tt).astype(int).reshape(D, Nx, Nz) + se[sidx - 1, 1].reshape(D, Nx, Nz)
    span = max((last[:, x:x + 16, z:z + 16].max(axis=(1, 2)) - first[:, x:x + 16, z:z + 16].min(axis=(1, 2))).max()
               for x in range(0, Nx, 16) for z in range(0, Nz, 16)) + 1
    assert rows - 64 < 3 * span + 1 <= rows or rows == 128 and 3 * span + 1 <= rows
    plan = DevicePlan(Nz, Nx, D, nT, R, tt, sir=(sidx, sir, se))
    sg = g.standard_normal((B, D, nT))
    ref = O.transpose_sir(np.transpose(sg, (0, 2, 1)), sidx.T, np.ascontiguousarray(tt.T), sir.T, se.T, R)
    sd = torch.tensor(sg, dtype=torch.float32).cuda()
    for v in (-1, 59, 60, 61, 62):
        plan.set_launch(B, v, 0)
        assert rel_l2(plan.transpose(sd, model=False).cpu().numpy().reshape(B, -1), ref) < TOL_OP, v


def test_one_sinogram_tile_variants_match_oracle():
    """Every one-sinogram tile form on a real arc geometry (the tile windows fit the LDS only
    for smooth travel times): forward choices 2, 3 (record streaming), 5, 6, 7 (tile form, thread
    per row), 9, 10 (its lean form) and 11, 12, 13 (the lean form over rows sorted by record
    count: the same sums as 9, bit for bit),
    gather variants 44-54 (LDS tile gathers, packed tile-major table), each against the
    oracle's DAS loops."""
    import torch
    _log("one-sinogram tile variants 96x80")
    m = _geometry_model(96, 80, 40, 700, 1e-4, sir=False, sigma=1.0)
    orc = _oracle_of(m)
    plan = m.plan
    D, nT = m.shape_sinogram
    x = rng(31).uniform(0, 1, (1, 80, 96))
    sg = rng(32).standard_normal((1, D, nT))
    tt = orc.tt.T   # [P x D]
    yo = np.transpose(O.forward_das(x.reshape(1, -1), tt, nT, orc.R), (0, 2, 1))
    xto = O.transpose_das(np.transpose(sg, (0, 2, 1)), tt, orc.R)
    xd = torch.tensor(x, dtype=torch.float32).cuda()
    sd = torch.tensor(sg, dtype=torch.float32).cuda()
    done = []
    ref = None
    for gv in range(44, 55):
        try:
            plan.set_launch(1, gv, 6)
        except Exception:
            continue
        xt = plan.transpose(sd, model=False).cpu().numpy()
        assert rel_l2(xt.reshape(1, -1), xto) < TOL_OP, gv
        if gv == 47:
            ref = xt
        if gv == 53:   # the packed table in 8 detector groups, as variant 47 (u rounded to 2^-23)
            assert ref is not None and rel_l2(xt, ref) < 1e-6
        done.append(gv)
    assert {47, 53}.issubset(done), done
    lean = None
    for ch in (2, 3, 5, 6, 7, 9, 10, 11, 12, 13):
        plan.set_launch(1, 47, ch)
        y = plan.forward(xd, model=False).cpu().numpy()
        assert rel_l2(y, yo) < TOL_OP, ch
        if ch == 9:
            lean = y
        if ch >= 10:   # chunk size, detector grouping and row order leave each row's sum unchanged
            assert np.array_equal(y, lean), ch
    plan.set_launch(1, -1, 0)


def _geometry_model(Nz, Nx, D, nT, h, sir=False, sigma=None):
    """Model with the benchmark geometry scaled down, built by the product setup code."""
    from mbrec.discretization import Discretization
    from mbrec.model import MSOTmodel
    from mbrec.probe import Probe
    half = (Nx - 1) / 2 * h
    disc = Discretization([-half, half, -(Nz - 1) / 2 * h, (Nz - 1) / 2 * h], [Nx, Nz])
    probe = Probe("arc256_r40_174", True, False, num_detectors=D)
    probe.DAC.numRecordedSamplesPerTransducer = nT
    # shift the recording window so the small field of view lands mid-sinogram
    probe.DAC.delayBeforeRecording = int(round(probe.detector.radius / 1500.0 * probe.DAC.frequency)) - nT // 2
    return MSOTmodel(probe, disc, 1500.0, sir, True, 0, 1e5, 12e6, sigma)


def _oracle_of(model):
    """Oracle model of the same acquisition.  Travel times, the interpolation radius and the
    SPMR indices are the oracle's own (restated from refraction.m:20-24, MSOTmodel.m:36-38,
    380-381, 472-478, 573-597 and Probe.m:112-115, pinned by hand-computed values), computed
    from the grid and probe parameters; the product's tables are only compared with them.
    The SIR table values, the IR and sigma are inputs (data) shared with the model; the
    prefilter kernels come from the oracle's own direct DFT of the Gaussian pixel
    (sigma = round(h/2 um), Discretization.m:43)."""
    d = model.Discretization
    Nz, Nx = d.Nz, d.Nx
    probe = model.Probe
    D = probe.detector.numOfTransducers
    c, fs = model.Medium.speedOfSound, probe.DAC.frequency
    X, Z = d.region["xPositionsFov"].T, d.region["zPositionsFov"].T
    xd, zd = O.arc_detectors(D, probe.detector.radius, probe.detector.angularCoverage)
    tt = O.travel_times(X, Z, xd, zd, c, fs, probe.DAC.delayBeforeRecording,
                        model.DataPreprocessing.numCroppedSamplesAtSinogramStart)
    np.testing.assert_allclose(model.Data.absoluteTravelTimeIndices.reshape(D, -1), tt, rtol=0, atol=1e-9)
    R = (Z[0, 1] - Z[0, 0]) * fs / c
    assert abs(R - model.Data.circularInterpolationRadiusInSamples) < 1e-12
    sig_px = d.pixelSigma   # the model's own sigma = round(min(dx, dz) / 2 um)
    kz, kx = O.full_kernels(Nz, Nx, d.dz, d.dx, sig_px)
    kw = dict(kz=kz, kx=kx, ir=model.Data.IR)
    if model.includeSir:
        g = model.Data.SPMRGrid
        sidx = O.spmr_indices(*O.spmr_polar(X, Z, xd, zd), g["dmin"], g["dd"], g["da"], g["n_angle"])
        np.testing.assert_array_equal(model.Data.SPMRIndices, sidx)
        kw.update(sidx=sidx.astype(np.int32), sir=model.Data.SPMR, se=model.Data.SPMRTimestepIndexStartAndEnd)
    return O.Model(Nz, Nx, tt, model.Data.numTimeSamplesPerTransducer, R, sigma=model.normalizationFactor, **kw)


def test_sigma_matches_dense_svd():
    """sigma_max of the unnormalised model (MSOTmodel.m:271-287, svds there) from the
    product's device power iteration equals the largest singular value of the oracle's
    dense FP64 operator (numpy SVD)."""
    _log("sigma vs dense SVD")
    m = _geometry_model(12, 10, 12, 160, 1.25e-4, sir=False, sigma=None)
    orc = _oracle_of(m)
    orc1 = O.Model(orc.Nz, orc.Nx, orc.tt, orc.nT, orc.R, sigma=1.0, kz=orc.kz, kx=orc.kx, ir=orc.ir)
    P = 12 * 10
    E = np.eye(P).reshape(P, 10, 12)
    A = orc1.forward(E).reshape(P, -1).T
    s_true = np.linalg.svd(A, compute_uv=False)[0]
    s_dev = m.estimate_sigma()
    assert abs(s_dev - s_true) / s_true < 1e-6, (s_dev, s_true)
    assert abs(m.normalizationFactor - s_true) / s_true < 1e-6


@pytest.mark.parametrize("per_det", [False, True])
def test_model_operators_generic_ir_length(per_det):
    """An IR of 57 taps (padded to 64, not the 201 taps the filter kernel is unrolled
    for) takes the IR filter with its tap count read at run time: the model forward and
    transpose against the oracle, one IR for all detectors or one per detector."""
    import torch
    from mbrec.model import DevicePlan
    _log(f"generic IR length per_det={per_det}")
    Nz, Nx, D, nT, R = 24, 20, 10, 300, 2.6666666666666665
    tt = random_tt(Nz * Nx, D, nT, R, seed=91, spill=0.05)
    ir = rng(92).standard_normal((D, 57) if per_det else 57)
    plan = DevicePlan(Nz, Nx, D, nT, R, tt.T, ir=ir)
    orc = O.Model(Nz, Nx, np.ascontiguousarray(tt.T), nT, R, ir=ir)
    x = rng(93).uniform(0, 1, (2, Nx, Nz))
    y = plan.forward(torch.tensor(x, dtype=torch.float32).cuda()).cpu().numpy()
    assert rel_l2(y.reshape(2, -1), orc.forward(x).reshape(2, -1)) < TOL_OP
    s = rng(94).standard_normal((2, D, nT))
    xt = plan.transpose(torch.tensor(s, dtype=torch.float32).cuda()).cpu().numpy()
    assert rel_l2(xt.reshape(2, -1), orc.transpose(s).reshape(2, -1)) < TOL_OP


@pytest.mark.parametrize("L,nT,D,B", [(1, 40, 3, 1), (15, 300, 5, 1), (33, 2053, 5, 1), (193, 190, 3, 2),
                                      (201, 2048, 7, 1), (207, 2053, 5, 3), (201, 300, 257, 2)])
def test_ir_filter_tap_split(L, nT, D, B):
    """The IR filter with its taps split over the parts of a workgroup (few rows): four parts for
    193..208 taps, two else, one group of taps only, records shorter than the taps, one and two
    tiles per record with a remainder; and the unsplit form above 511 tiles.  FP64 sums of FP32
    samples: the other operator tests' limit."""
    import torch
    from mbrec.model import DevicePlan
    _log(f"IR filter split L={L} nT={nT} D={D} B={B}")
    Nz, Nx, R = 12, 10, 2.6666666666666665
    tt = random_tt(Nz * Nx, D, nT, R, seed=L + nT, spill=0.05)
    ir = rng(L).standard_normal(L)
    plan = DevicePlan(Nz, Nx, D, nT, R, tt.T, ir=ir)
    orc = O.Model(Nz, Nx, np.ascontiguousarray(tt.T), nT, R, ir=ir)
    x = rng(95).uniform(0, 1, (B, Nx, Nz))
    y = plan.forward(torch.tensor(x, dtype=torch.float32).cuda()).cpu().numpy()
    assert rel_l2(y.reshape(B, -1), orc.forward(x).reshape(B, -1)) < TOL_OP
    s = rng(96).standard_normal((B, D, nT))
    xt = plan.transpose(torch.tensor(s, dtype=torch.float32).cuda()).cpu().numpy()
    assert rel_l2(xt.reshape(B, -1), orc.transpose(s).reshape(B, -1)) < TOL_OP


@pytest.mark.parametrize("fir_mfma", [True, False])
@pytest.mark.parametrize("sir", [False, True])
def test_model_operators_match_oracle(sir, fir_mfma):
    """Both IR filter kernels (FP64 matrix cores, vector) against the oracle, with the
    adjoint identity of the device pair."""
    import torch
    _log(f"model_ops sir={sir} fir_mfma={fir_mfma}")
    m = _geometry_model(48, 40, 32, 700, 1e-4, sir=sir, sigma=2.5)
    m.plan.set_fir_kernel(fir_mfma)
    orc = _oracle_of(m)
    x = np.maximum(rng(9).standard_normal((2, 40, 48)), 0)
    y = m.applyForward(x)
    yo = orc.forward(x)
    assert rel_l2(y, yo) < TOL_OP, rel_l2(y, yo)
    s = rng(10).standard_normal((2, 32, 700))
    xt = m.applyTranspose(s)
    assert rel_l2(xt, orc.transpose(s)) < TOL_OP
    # adjoint identity of the device pair, FP64 inner products of FP32 results
    xd = torch.tensor(x, dtype=torch.float32).cuda()
    sd = m.applyForward(torch.tensor(np.maximum(rng(11).standard_normal((2, 40, 48)), 0), dtype=torch.float32).cuda())
    lhs = torch.sum(m.applyForward(xd).double() * sd.double()).item()
    rhs = torch.sum(xd.double() * m.applyTranspose(sd).double()).item()
    assert abs(lhs - rhs) <= TOL_ADJ * abs(lhs), (lhs, rhs)


def test_nnls_L2_matches_oracle():
    import torch
    from mbrec.solvers import rec_nn_with_L2_reg
    from mbrec.phantoms import disks, add_noise
    _log("nnls_L2 parity")
    m = _geometry_model(40, 40, 32, 600, 1.25e-4, sir=False, sigma=3.0)
    orc = _oracle_of(m)
    ph = np.stack([disks(m.Discretization, n=6, seed=s) for s in (1, 2)])
    y = add_noise(orc.forward(ph), 0.01, seed=3)
    lam = 1e-2 * np.linalg.norm(orc.transpose(y))
    for coupled in (True, False):
        rec, e_img, e_reg, *_ = rec_nn_with_L2_reg(m, y, 20, lam, coupled=coupled)
        if coupled:
            ro, lc, _ = orc.rec_nn_with_L2_reg(y, 20, lam)
            assert rel_l2(rec, ro) < TOL_REC
            assert abs(e_img - lc[0]) < 1e-3 * lc[0]
        else:
            for w in range(2):
                ro, lc, _ = orc.rec_nn_with_L2_reg(y[w:w + 1], 20, lam)
                assert rel_l2(rec[w], ro) < TOL_REC
                assert abs(e_img[w] - lc[0]) < 1e-3 * lc[0]


def test_nnls_warm_start_seeds_outer_iterate():
    """init really seeds w0 (the hook the learned warm start uses): with 0 outer
    iterations the result is the seed itself, without a seed it is zero."""
    import torch
    from mbrec.solvers import rec_nn_with_L2_reg
    m = _geometry_model(24, 24, 16, 400, 1.25e-4, sir=False, sigma=3.0)
    y = rng(12).standard_normal((2, 16, 400))
    seed = rng(13).uniform(0, 1, (2, 24, 24)).astype(np.float32)
    r0, *_ = rec_nn_with_L2_reg(m, y, 0, 0.0, coupled=False, init=seed)
    np.testing.assert_array_equal(r0.astype(np.float32), seed)
    z0, *_ = rec_nn_with_L2_reg(m, y, 0, 0.0, coupled=False)
    assert not np.any(z0)


def test_nnls_L1_matches_oracle():
    from mbrec.solvers import rec_nn_with_L1_eye_reg
    from mbrec.phantoms import disks, add_noise
    _log("nnls_L1 parity")
    m = _geometry_model(40, 40, 32, 600, 1.25e-4, sir=False, sigma=None)
    orc = _oracle_of(m)
    ph = np.stack([disks(m.Discretization, n=6, seed=s) for s in (5, 6)])
    y = add_noise(orc.forward(ph), 0.01, seed=7)
    eta = 0.05 * np.abs(orc.transpose(y)).max()     # a shrinkage that leaves a non-trivial image
    for coupled in (True, False):
        rec, e_img, e_reg, *_ = rec_nn_with_L1_eye_reg(m, y, 15, eta, coupled=coupled)
        if coupled:
            ro, _ = orc.rec_nn_with_L1_eye_reg(y, 15, eta)
            assert rel_l2(rec, ro) < TOL_REC
        else:
            for w in range(2):
                ro, _ = orc.rec_nn_with_L1_eye_reg(y[w:w + 1], 15, eta)
                assert rel_l2(rec[w], ro) < TOL_REC


def test_nnls_warm_start_dual_matches_oracle():
    """The warm-start form (outer iterate w0 and scaled dual v0 of nnls_L2_less) against the
    oracle started from the same pair, independent solves with their own lambdaL2."""
    import torch
    from mbrec.solvers import rec_nn_with_L2_reg_batch
    from mbrec.phantoms import disks, add_noise
    _log("nnls_L2 warm start (w0, v0)")
    m = _geometry_model(24, 24, 16, 400, 1.25e-4, sir=False, sigma=3.0)
    orc = _oracle_of(m)
    ph = np.stack([disks(m.Discretization, n=4, seed=s) for s in (5, 6)])
    y = add_noise(orc.forward(ph), 0.01, seed=7)
    lam = [1e-2 * np.linalg.norm(orc.transpose(y[b:b + 1])) for b in range(2)]
    g = rng(8)
    w0 = np.maximum(g.standard_normal((2, 24, 24)), 0) * np.abs(ph).max()
    v0 = g.standard_normal((2, 24, 24)) * np.abs(ph).max()
    got = rec_nn_with_L2_reg_batch(m, torch.as_tensor(y, dtype=torch.float32).cuda(), 10, lam,
                                   init=w0.astype(np.float32), init_dual=v0.astype(np.float32)).cpu().numpy()
    want = orc.rec_nn_with_L2_reg_from(y, 10, lam, w0, v0)
    cold = orc.rec_nn_with_L2_reg_from(y, 10, lam)
    assert rel_l2(want, cold) > 1e-2          # the start matters
    assert rel_l2(got, want) < TOL_REC


def test_warm_start_state_training_and_fallback():
    """The warm-start machinery on a small geometry: device training lowers the loss; the
    loop started from the stationary state s* of the minimiser (the network's target:
    w0 = max(s*, 0), v0 = max(-s*, 0)) stays at the minimiser, where the cold start is still
    away from it; a network output that is not finite, or whose image scores a larger
    objective than the cold start, is replaced by the cold start.  The gain of the trained
    400^2 network is measured at full size (test_full_size.py)."""
    import torch
    from mbrec.solvers import rec_nn_with_L2_reg_batch
    from mbrec.warmstart import (UNet, make_training_set, nnls_l2_minimiser, phantom_batch, stationary_state,
                                 train, warm_start_estimate)
    _log("warm start: training, state form, fallback")
    # sigma_max-normalised model: the minimiser's step 1/L assumes ||A|| <= 1
    m = _geometry_model(32, 32, 16, 400, 1.25e-4, sir=False, sigma=None)
    xin, xt = make_training_set(m, 64, 500, batch=32)
    net = UNet(32, seed=1)
    hist = train(net, xin, xt, epochs=25, batch=8, lr=2e-3, seed=1)
    assert hist[-1] < 0.5 * hist[0]
    ph = torch.as_tensor(phantom_batch(m.Discretization, 8, 9000)).cuda()
    y = m.applyForward(ph)
    gen = torch.Generator(device="cuda").manual_seed(3)
    y = (y + 0.01 * y.abs().amax(dim=(1, 2), keepdim=True) * torch.randn(y.shape, generator=gen,
                                                                           device="cuda")).contiguous()
    lam = (1e-2 * torch.linalg.vector_norm(m.applyTranspose(y).reshape(8, -1).double(), dim=1)).cpu().numpy()
    ref, kkt = nnls_l2_minimiser(m, y, lam)
    assert kkt < 1e-6
    nref = torch.linalg.vector_norm(ref.reshape(8, -1).double(), dim=1)

    def err(r):
        return float((torch.linalg.vector_norm((r.double() - ref).reshape(8, -1), dim=1) / nref).max())

    k = 5
    s = stationary_state(m, y, lam, ref)
    w0, v0 = torch.clamp(s, min=0.0).float().contiguous(), torch.clamp(-s, min=0.0).float().contiguous()
    e_state = err(rec_nn_with_L2_reg_batch(m, y, k, lam, init=w0, init_dual=v0))
    e_cold = err(rec_nn_with_L2_reg_batch(m, y, k, lam))
    print(f"worst error after {k} iterations: from s* {e_state:.2e}, cold {e_cold:.2e}", flush=True)
    assert e_state < 1e-5 and e_cold > 100 * e_state

    class Fixed:
        def __init__(self, out):
            self.out = out

        def forward(self, aty):
            return self.out

    bad = torch.zeros((8, 32, 32), dtype=torch.float32, device="cuda")
    bad[0, 3, 3] = float("nan")
    bad[1] = 1e6                    # a huge image: larger objective than w = 0
    bad[2:] = s[2:].float()
    w0, v0, used = warm_start_estimate(Fixed(bad), m, y, lam)
    assert not used[0] and not used[1] and used[2:].all()
    assert float(w0[:2].abs().max()) == 0.0 and float(v0[:2].abs().max()) == 0.0
    assert torch.equal(w0[2:], torch.clamp(bad[2:], min=0.0))
    # the cold start as arbiter: exact states are kept, a finite state with a huge dual (it
    # passes the objective test: its image is 0) loses to the cold start after 10 iterations
    from mbrec.warmstart import arbitrate_warm_start
    v_bad = v0.clone()
    v_bad[3] = 1e4 * float(v0[2:].abs().max())
    wj, vj, keep = arbitrate_warm_start(m, y, lam, w0, v_bad, used, k=10)
    assert not keep[0] and not keep[1] and not keep[3] and keep[2] and keep[4:].all()
    wc, vc = rec_nn_with_L2_reg_batch(m, y, 10, lam, return_dual=True)
    assert torch.equal(wj[3], wc[3]) and torch.equal(vj[3], vc[3])
    # the learned solve chains estimate, fallback, arbiter and the remaining iterations
    from mbrec.warmstart import rec_nn_with_L2_reg_learned
    rec_l, used_l = rec_nn_with_L2_reg_learned(Fixed(bad), m, y, 15, lam, arbiter_iters=10)
    w0, v0, used = warm_start_estimate(Fixed(bad), m, y, lam)
    wa, va, ka = arbitrate_warm_start(m, y, lam, w0, v0, used, k=10)
    assert torch.equal(rec_l, rec_nn_with_L2_reg_batch(m, y, 5, lam, init=wa, init_dual=va))
    assert np.array_equal(used_l, ka)
