"""The fused step of models with 25 to 128 dofs: one substep from identical state against the per-stage step. The sizes and
orders are those where the dense solver's bookkeeping (row masks, short rows staged by their columns, the packed Hessian)
can go wrong: the smallest and the largest dof count, bodies apart, in chains and all in contact, rows of every kind
(connect, weld, joint equality, friction loss, contact, limit), dofs in both halves of the wavefront, and one, two and four
environments per workgroup (the packed Hessian of the largest models is in LDS with one, in the state record with more)."""

from __future__ import annotations

import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from genesis_amd import scenes
from genesis_amd.model.compiler import SolverOptions, compile_model
from genesis_amd.model.mjcf import load_mjcf
from genesis_amd.model.primitives import box_entity, plane_entity, sphere_entity
from tests.parity import check_fused_matches_plain

pytestmark = pytest.mark.gpu

ARM = """<mujoco model="arm"><worldbody><body name="a" pos="{x} 0 0.3">
  <joint name="j1" type="hinge" axis="0 1 0" range="-0.3 0.3" limited="true" frictionloss="0.2"/>
  <inertial pos="0.1 0 0" mass="1" diaginertia="0.01 0.02 0.03"/>
  <geom type="capsule" fromto="0 0 0 0.2 0 0" size="0.04"/>
  <body name="b" pos="0.2 0 0"><joint name="j2" type="slide" axis="1 0 0" range="-0.05 0.05" limited="true"/>
    <inertial pos="0.1 0 0" mass="0.5" diaginertia="0.01 0.02 0.03"/>
    <geom type="sphere" size="0.06" pos="0.1 0 0"/></body></body></worldbody>
  <equality><joint joint1="j1" joint2="j2" polycoef="0.02 0.5 0 0 0"/></equality></mujoco>"""


def _boxes(n, spacing, opts):
    """n free boxes with their centres ``spacing`` apart on a line, alternating with spheres."""
    ents = [plane_entity(friction=0.5)]
    for i in range(n):
        pos = np.array([spacing * i, 0.01 * (i % 3), 0.049])
        if i % 4 == 3:
            ents.append(sphere_entity(0.05, pos, np.array([1.0, 0, 0, 0]), rho=500.0, friction=0.5, name=f"s{i}"))
        else:
            ents.append(box_entity(np.full(3, 0.1), pos, np.array([1.0, 0, 0, 0]), rho=500.0, friction=0.5, name=f"b{i}"))
    return compile_model(ents, SolverOptions(dt=0.01, **opts))


def _arms(tmp_path, n, opts):
    ents = [plane_entity()]
    for i in range(n):
        p = os.path.join(str(tmp_path), f"arm{i}.xml")
        with open(p, "w") as f:
            f.write(ARM.format(x=0.33 * i))
        ents.append(load_mjcf(p, f"arm{i}"))
    return compile_model(ents, SolverOptions(dt=0.01, **opts))


def _loops(tmp_path, n, opts):
    return compile_model([load_mjcf(scenes.CLOSED_LOOPS_XML, f"l{i}") for i in range(n)], SolverOptions(dt=0.005, **opts))


def _quads(tmp_path, n, opts):
    return compile_model([plane_entity()] + [load_mjcf(scenes.QUADRUPED_XML, f"q{i}") for i in range(n)],
                         SolverOptions(dt=0.005, **opts))


MODELS = {
    "boxes_apart_30": lambda t, o: _boxes(5, 0.5, o),  # bodies apart
    "boxes_touching_30": lambda t, o: _boxes(5, 0.099, o),  # one chain of contacts
    "boxes_pairs_126": lambda t, o: _boxes(21, 0.0995, o),  # one chain over both halves of the wavefront
    "boxes_pairs_132": lambda t, o: _boxes(22, 0.0995, o),  # more dofs than two per lane: no matrix cores
    "arms_26": lambda t, o: _arms(t, 13, o),  # friction, joint equality, limit and contact rows; two-dof entities
    "arms_128": lambda t, o: _arms(t, 64, o),  # every position of a lane used
    "loops_30": lambda t, o: _loops(t, 3, o),  # connect and weld rows
    "boxes_touching_48": lambda t, o: _boxes(8, 0.099, o),  # the most dofs whose private region fits in LDS, about
    "quadrupeds_36": lambda t, o: _quads(t, 2, o),  # overlapping robots: long rows, 18-dof entities
}


# "alone": no collisions (boxes then have no rows); the detections differ for pairs of boxes only
OPTIONS = {"sat": {"box_box_detection": True}, "mpr": {"box_box_detection": False}, "alone": {"enable_collision": False}}


def _one_step_equals_the_per_stage_step(model, name, opts, config):
    from genesis_amd import runtime as rt

    rt.load_library()
    assert model.n_dofs > 24
    dm = rt.DeviceModel(model)
    if config is not None:
        dm.set_fused_config(*config)
    B = 17
    a = rt.StateSlab(dm, B)
    gen = torch.Generator().manual_seed(5)
    a["vel"].copy_(0.3 * torch.randn(model.n_dofs, B, generator=gen))
    if name.startswith("arms"):
        a["qpos"].copy_(0.4 * torch.randn(model.n_qs, B, generator=gen))
    a.forward_kinematics()
    a.step(3, rt.RS_MODE_PLAIN)
    torch.cuda.synchronize()
    b = rt.StateSlab(dm, B)
    b.buffer.copy_(a.buffer)
    print(f"[islands] {name} D={model.n_dofs} rows up to {int(a['n_con'].max())} config={dm.fused_config}", flush=True)
    a.step(1, rt.RS_MODE_PLAIN)
    b.step(1, rt.RS_MODE_FUSED)
    torch.cuda.synchronize()
    assert int(a["n_con"].max()) > 0 or (name, opts) == ("quadrupeds_36", "alone")  # no joint past its limit
    check_fused_matches_plain(a, b, model)
    return dm.fused_config


@pytest.mark.parametrize("epb", [1, 2, 4])
@pytest.mark.parametrize("name, opts", [(n, o) for n in MODELS for o in OPTIONS if (o != "alone" or "boxes" not in n) and n != "boxes_pairs_132"])
def test_island_step_matches_the_per_stage_step(tmp_path, name, opts, epb):
    _one_step_equals_the_per_stage_step(MODELS[name](tmp_path, OPTIONS[opts]), name, opts, (epb, False, False, 0))


@pytest.mark.parametrize("name, opts, in_lds", [
    ("arms_26", "mpr", True), ("loops_30", "alone", True), ("boxes_touching_30", "sat", True),
    ("quadrupeds_36", "mpr", True), ("boxes_touching_48", "sat", True), ("boxes_touching_48", "mpr", True),
    ("boxes_pairs_126", "sat", False), ("arms_128", "alone", False), ("boxes_pairs_132", "sat", False)])
def test_default_launch_shape_matches_the_per_stage_step(tmp_path, name, opts, in_lds):
    """As a model is created: one environment per workgroup, the private region in LDS where it fits."""
    c = _one_step_equals_the_per_stage_step(MODELS[name](tmp_path, OPTIONS[opts]), name, opts, None)
    assert c["envs_per_block"] == 1 and c["use_lds"] == in_lds


def test_nan_pose_stays_in_its_environment(tmp_path):
    """A NaN pose makes a weld's rows NaN in every column, also in those of bodies it does not join. Its environment
    reports the error; its neighbours come out bit for bit as without it."""
    from genesis_amd import runtime as rt

    rt.load_library()
    model = MODELS["loops_30"](tmp_path, OPTIONS["alone"])
    dm = rt.DeviceModel(model)
    slabs = []
    for bad in (False, True):
        s = rt.StateSlab(dm, 9)
        gen = torch.Generator().manual_seed(3)
        s["vel"].copy_(0.3 * torch.randn(model.n_dofs, 9, generator=gen))
        s.forward_kinematics()
        if bad:
            s["links_quat"][:, 4] = float("nan")
        print(f"[islands] loops_30 NaN pose in env 4: {bad}", flush=True)
        s.step(1, rt.RS_MODE_FUSED)
        torch.cuda.synchronize()
        slabs.append(s)
    good, bad = slabs
    rest = [b for b in range(9) if b != 4]
    assert int(bad["n_con"].max()) > 0
    for name in ("qpos", "vel", "acc", "links_pos", "efc_force", "errbits"):
        assert torch.equal(good[name][:, rest], bad[name][:, rest]), name
    assert int(bad["errbits"][0, 4]) & rt.ERR_INVALID_FORCE_NAN


@pytest.mark.parametrize("name, in_lds", [("boxes_apart_30", True), ("boxes_apart_30", False), ("boxes_pairs_126", False)])
def test_nan_velocity_spreads_as_in_the_per_stage_step(tmp_path, name, in_lds):
    """Products leave out the tiles in which every row is zero, where a row force that is not a number would have added one:
    the environment's accelerations, forces and error bits are those of the per-stage step all the same."""
    from genesis_amd import runtime as rt

    rt.load_library()
    model = MODELS[name](tmp_path, OPTIONS["sat"])
    dm = rt.DeviceModel(model)
    dm.set_fused_config(1, in_lds, False, 0)
    a = rt.StateSlab(dm, 5)
    gen = torch.Generator().manual_seed(5)
    a["vel"].copy_(0.3 * torch.randn(model.n_dofs, 5, generator=gen))
    a.forward_kinematics()
    a.step(3, rt.RS_MODE_PLAIN)
    torch.cuda.synchronize()
    a["vel"][model.n_dofs - 2, 2] = float("nan")
    b = rt.StateSlab(dm, 5)
    b.buffer.copy_(a.buffer)
    print(f"[islands] {name} NaN velocity of the last body in env 2, config={dm.fused_config}", flush=True)
    a.step(1, rt.RS_MODE_PLAIN)
    b.step(1, rt.RS_MODE_FUSED)
    torch.cuda.synchronize()
    assert torch.equal(a["errbits"], b["errbits"]) and int(b["errbits"][0, 2]) & rt.ERR_INVALID_FORCE_NAN
    for field in ("acc", "qacc_ws", "qf_constraint", "vel", "qpos"):
        assert torch.equal(a[field].isnan(), b[field].isnan()), field
    assert torch.equal(a["qpos"][:, 2], b["qpos"][:, 2])  # the NaN guard kept the old pose


@pytest.mark.parametrize("n_small", [33, 2100])
def test_shared_launch_of_both_classes_equals_the_launches_alone(tmp_path, n_small):
    """Row-tile models and larger ones (region in LDS when alone, collision-free, the most dofs of the matrix-core path, and
    beyond it) in one shared step: bit for bit the steps of each alone, with only the caller's stream to wait for. With few
    small environments the step is one launch, with 4200 quadrupeds it is two on two streams."""
    from genesis_amd import runtime as rt

    rt.load_library()
    models = [scenes.franka_model(), _boxes(5, 0.099, OPTIONS["sat"]), _boxes(22, 0.0995, OPTIONS["sat"]),
              scenes.quadruped_model(), _loops(tmp_path, 3, OPTIONS["alone"]), _arms(tmp_path, 64, OPTIONS["alone"])]
    assert [m.n_dofs for m in models] == [9, 30, 132, 18, 30, 128]
    sizes = [n_small, 9, 5, 2 * n_small, 7, 3]
    alone, mixed = [], []
    for m, n in zip(models, sizes):
        dm = rt.DeviceModel(m)
        a = rt.StateSlab(dm, n)
        gen = torch.Generator().manual_seed(n)
        a["vel"].copy_(0.2 * torch.randn(m.n_dofs, n, generator=gen))
        a.forward_kinematics()
        b = rt.StateSlab(dm, n)
        b.buffer.copy_(a.buffer)
        alone.append(a)
        mixed.append(b)
    torch.cuda.synchronize()
    shared, stream = rt.SharedLaunch(8), torch.cuda.Stream()
    got = []
    for step in range(6):  # more steps than segment tables; every step's outputs are read on the caller's stream alone
        with torch.cuda.stream(stream):
            shared.step(mixed, stream)
            got.append([s["vel"].clone() for s in mixed])
    stream.synchronize()
    for step in range(6):
        for a, g in zip(alone, got[step]):
            a.step(1, rt.RS_MODE_FUSED)
            torch.cuda.synchronize()
            assert torch.equal(a["vel"], g), (a.dmodel.model.n_dofs, step)
    for a, b in zip(alone, mixed):
        for name in ("qpos", "acc", "n_con", "errbits"):
            assert torch.equal(a[name], b[name]), (a.dmodel.model.n_dofs, name)
    assert all(int(b["n_con"].max()) > 0 for b in mixed[1:])


def _frames(tmp_path, n):
    """n bodies without joints, one entity."""
    p = os.path.join(str(tmp_path), f"frames{n}.xml")
    with open(p, "w") as f:
        f.write('<mujoco model="frames"><worldbody><body name="r" pos="5 0 0">')
        for i in range(n):
            f.write(f'<body name="f{i}" pos="0 {0.01 * i} 0"><inertial pos="0 0 0" mass="0.1" '
                    'diaginertia="0.001 0.001 0.001"/></body>')
        f.write("</body></worldbody></mujoco>")
    return load_mjcf(p, "frames")


@pytest.mark.parametrize("n_links", [64, 900])
def test_rows_are_built_dense_where_their_staging_does_not_fit(tmp_path, n_links):
    """Four environments per workgroup, contact rows staged with four LDS words per link: with 900 links that does not fit,
    and the launch is accepted all the same."""
    ents = [plane_entity(friction=0.5), _frames(tmp_path, n_links)]
    for i in range(5):
        ents.append(box_entity(np.full(3, 0.1), np.array([0.099 * i, 0.01 * (i % 3), 0.049]), np.array([1.0, 0, 0, 0]),
                               rho=500.0, friction=0.5, name=f"b{i}"))
    model = compile_model(ents, SolverOptions(dt=0.01, box_box_detection=True))
    assert model.n_links > n_links and model.n_dofs == 30
    c = _one_step_equals_the_per_stage_step(model, "boxes", "sat", (4, False, False, 0))
    assert c["envs_per_block"] == 4 and not c["use_lds"] and 4 * c["lds_bytes_per_env"] <= 65536


def test_update_refuses_a_tree_with_longer_chains():
    """Launches stage rows of as many dofs as two of the created model's chains have; a box hung under another would double
    them. Other values are updated as before."""
    from genesis_amd import runtime as rt

    rt.load_library()
    model = _boxes(5, 0.5, OPTIONS["sat"])
    dm = rt.DeviceModel(model)
    parent = model.arrays["link_parent"]
    keep = parent.copy()
    parent[3] = 2
    with pytest.raises(rt.RigidStepError, match="longer chains"):
        dm.update()
    parent[:] = keep
    model.arrays["geom_friction"][:] = 0.7
    dm.update()
