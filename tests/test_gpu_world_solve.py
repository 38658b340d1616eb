"""The per-world solve of the forms it takes besides plain TGS piles (PGS
passes, joints with limits, sleeping), in both workgroup shapes (a world a wave
when worlds fill the chip, four waves when they do not) and with records in LDS
or in HBM, against one launch per colour and iteration: the same bits."""
import numpy as np
import pytest

import physx_amd as P
from physx_amd import scenes as S

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0


def _piles(n):
    return S.batched_piles(n_scenes=n, nmin=8, nmax=96 if n > 100 else 300, seed=21)


def _chains(n):
    return S.jointed_chains(n_scenes=n, links=5, drops=3, seed=6)


@pytest.mark.parametrize("lds", [None, 0, 40])
@pytest.mark.parametrize("kind,worlds,kw", [
    ("piles", 24, dict(solver_type=P.PXH_SOLVER_PGS)), ("piles", 1100, dict(solver_type=P.PXH_SOLVER_PGS)),
    ("piles", 24, dict(enable_sleeping=1)), ("chains", 8, {}), ("chains", 1040, {}),
    ("chains", 8, dict(enable_sleeping=1))])
def test_world_solve_forms(cuda, kind, worlds, kw, lds):
    sc = _piles(worlds) if kind == "piles" else _chains(8)
    if kind == "chains" and worlds > 8:
        # copies of the eight worlds, enough of them to fill the chip
        per = sc.n // 8
        rep = worlds // 8
        j, k = sc.joints, len(sc.joints["type"])
        shift = np.repeat(np.arange(rep) * sc.n, k)
        joints = {"type": np.tile(j["type"], rep), "frame0": np.tile(j["frame0"], (rep, 1)),
                  "frame1": np.tile(j["frame1"], (rep, 1))}
        for b in ("body0", "body1"):
            t = np.tile(j[b], rep)
            joints[b] = np.where(t >= 0, t + shift, -1).astype(np.int32)
        big = S.Scene(*(np.concatenate([a] * rep) for a in (sc.shape_type, sc.dims, sc.pose, sc.lin_vel, sc.ang_vel,
                                                            sc.mass, sc.inertia)),
                      np.repeat(np.arange(worlds, dtype=np.int32), per), np.concatenate([sc.planes] * rep),
                      np.arange(worlds, dtype=np.int32), worlds, "chains", {})
        big.joints = joints
        sc = big
    a = P.Scene(sc, position_iterations=4, velocity_iterations=1, **kw)
    a.set_tuning(layout=P.PXH_SOLVE_LAYOUT_COLORS)
    b = P.Scene(sc, position_iterations=4, velocity_iterations=1, **kw)
    if lds is not None:
        b.set_tuning(layout=P.PXH_SOLVE_LAYOUT_WORLDS, lds_bodies=lds)
    for _ in range(25):
        a.step(DT)
        b.step(DT)
    assert b.stats()["solve_launches"] == 1 and a.stats()["solve_launches"] > 1
    assert a.stats()["constraints"] == b.stats()["constraints"] > 0
    for x, y, name in zip(b.bodies(), a.bodies(), ("pose", "linear velocity", "angular velocity")):
        np.testing.assert_array_equal(x, y, err_msg=name)


def test_worlds_added_after_joints(cuda):
    """bodies added after a step with joints: the joint lists grow with the worlds"""
    one = _chains(4)
    late = S.batched_piles(n_scenes=2, nmin=20, nmax=30, seed=2)
    late.scene_id = late.scene_id + 4
    late.plane_scene = late.plane_scene + 4
    scenes = []
    for layout in (P.PXH_SOLVE_LAYOUT_COLORS, P.PXH_SOLVE_LAYOUT_WORLDS):
        s = P.Scene(one, position_iterations=4, velocity_iterations=1)
        s.set_tuning(layout=layout)
        s.step(DT, 5)
        s.add(late)
        s.step(DT, 10)
        scenes.append(s)
    for x, y in zip(scenes[1].bodies(), scenes[0].bodies()):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("lds", [None, 0])
@pytest.mark.parametrize("bodies", [65, 257, 500, 1023, 1024])
def test_pgs_motion_of_large_worlds(cuda, bodies, lds):
    """PGS worlds with several bodies a thread, the last wave of them partly
    idle: the motion saved after the position passes is that of the position
    passes, before any velocity pass changes it."""
    sc = S.batched_piles(n_scenes=4, nmin=bodies, nmax=bodies, seed=bodies)
    kw = dict(position_iterations=4, velocity_iterations=2, solver_type=P.PXH_SOLVER_PGS)
    a, b = P.Scene(sc, **kw), P.Scene(sc, **kw)
    a.set_tuning(layout=P.PXH_SOLVE_LAYOUT_COLORS)
    if lds is not None:
        b.set_tuning(layout=P.PXH_SOLVE_LAYOUT_WORLDS, lds_bodies=lds)
    for _ in range(40):
        a.step(DT)
        b.step(DT)
    assert b.stats()["solve_launches"] == 1 < a.stats()["solve_launches"]
    assert a.stats()["constraints"] > bodies
    for x, y, name in zip(b.bodies(), a.bodies(), ("pose", "linear velocity", "angular velocity")):
        np.testing.assert_array_equal(x, y, err_msg=name)
