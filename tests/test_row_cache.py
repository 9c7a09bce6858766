"""The sweeps' LDS record cache against the oracle, bit for bit, where a contact's record changes
place: all contacts in LDS, the last ones in global memory, and more contacts than one response
pass takes (21); an articulation on static geometry only, so the sweeps are one chain."""

import numpy as np
import pytest

import metalrobo as mr
import model_util as mu
import oracle_lib as ol

BOX, PLANE = 2, 3


def flat_chain(boxes, mass=None):
    """A floating chain of box links lying on a plane: four contacts a link. `mass(i)` replaces link i's mass."""
    def link(i, m, inertia, **joint):
        if mass is not None:
            m, inertia = mass(i), [mass(i) * x for x in (0.01, 0.012, 0.014)]
        return mu.body(m, inertia, **joint)

    links = [link(0, 2.0, [0.02] * 3)]
    shapes = [mu.shape(0, BOX, (0.1, 0.1, 0.05))]
    dofs = [mu.dof(0, mu.INVALID) for _ in range(6)]
    for i in range(1, boxes):
        links.append(link(i, 1.0 + 0.1 * i, [0.01, 0.012, 0.014], parent=i - 1, joint_type=0, q_index=6 + i,
                          v_index=5 + i, axis=(0, 1, 0), parent_anchor=(0.12, 0, 0), child_anchor=(-0.12, 0, 0)))
        dofs.append(mu.dof(i, 6 + i, drive=(0, 0, 0.02, 0)))
        shapes.append(mu.shape(i, BOX, (0.1, 0.1, 0.05)))
    ground = mu.body(0.0, [1, 1, 1], motion=0)
    shapes.append(mu.shape(boxes, PLANE, [], rot=mu.Y_TO_Z))
    return mu.CustomWorld(links + [ground], dofs, shapes, link_count=boxes, root_type=1, nq=6 + boxes, nv=5 + boxes,
                          envs=2)


@pytest.mark.gpu
@pytest.mark.parametrize("tolerance", [0.0, 1.0e-5])
@pytest.mark.parametrize("boxes", [1, 3, 6, 16])
def test_rows_in_lds_and_in_global_memory_match_oracle(gpu, boxes, tolerance):
    w = flat_chain(boxes)
    cfg = w.config(pair_capacity=128, manifold_capacity=64, constraint_capacity=96, residual_tolerance=tolerance)
    world, ost = mr.World(w.model, cfg), ol.OracleState(w.model, cfg)
    rng = np.random.default_rng(boxes)
    q = np.zeros((w.envs, w.nq), np.float32)
    q[:, 2], q[:, 6] = 0.0495, 1.0
    v = rng.uniform(-0.2, 0.2, (w.envs, w.nv)).astype(np.float32)
    scene = np.zeros((w.envs, 1), mr.BODY_STATE_DTYPE)
    scene[:] = mu.scene_state((0, 0, 0), motion=0)
    ost.q[:], ost.v[:], ost.scene[:] = q, v, scene
    world.set_state(q, v, scene)
    cmd = (0.3 * rng.standard_normal((5, w.envs, w.nv))).astype(np.float32)
    for k in range(len(cmd)):
        status, cs = ost.step(cmd[k], control_step=k)[:2]
        world.advance(cmd[k:k + 1])
        np.testing.assert_array_equal(world.statuses()[0]["code"], status["code"])
        assert np.all(status["code"] == 0) and int(cs["constraints"].min()) >= 2 * boxes
        np.testing.assert_array_equal(world.contact_statuses()[0]["residuals"].view(np.uint32),
                                      cs["residuals"].view(np.uint32))
        gq, gv, _ = world.state()
        assert np.array_equal(gq.view(np.uint32), ost.q.view(np.uint32)), k
        assert np.array_equal(gv.view(np.uint32), ost.v.view(np.uint32)), k


@pytest.mark.gpu
@pytest.mark.parametrize("heavy,fails_at", [(1, 5), (3, 13), (14, 57)])
def test_a_non_finite_update_reports_its_contact_in_lds_and_in_global_memory(gpu, heavy, fails_at):
    """A chain of light boxes and a heavy one falls at 1e37 m/s: an impulse of the heavy box overflows in
    the first sweep, at a contact whose record is in LDS (about the first nine are) or behind them. The
    oracle counts sweeps and takes residuals only after they all passed."""
    boxes = 16
    w = flat_chain(boxes, lambda i: 100.0 if i == heavy else 0.2)
    cfg = w.config(pair_capacity=128, manifold_capacity=64, constraint_capacity=96)
    world, ost = mr.World(w.model, cfg), ol.OracleState(w.model, cfg)
    q, v = np.zeros((w.envs, w.nq), np.float32), np.zeros((w.envs, w.nv), np.float32)
    q[:, 2], q[:, 6], v[:, 2] = 0.0495, 1.0, -1.0e37
    scene = np.zeros((w.envs, 1), mr.BODY_STATE_DTYPE)
    scene[:] = mu.scene_state((0, 0, 0), motion=0)
    ost.q[:], ost.v[:], ost.scene[:] = q, v, scene
    world.set_state(q, v, scene)
    cmd = np.zeros((w.envs, w.nv), np.float32)
    status, cs = ost.step(cmd, control_step=0)[:2]
    assert np.all(status["code"] != 0) and np.all(status["failing_index"] == fails_at), status["failing_index"]
    assert np.all(cs["solver_iterations"] == 0) and np.all(cs["constraints"] == 4 * boxes)
    world.advance(cmd[None])
    got = world.statuses()[0]
    for f in ("code", "failing_index", "successful_substeps"):
        np.testing.assert_array_equal(got[f], status[f], err_msg=f)
    np.testing.assert_array_equal(world.contact_statuses()[0]["constraints"], cs["constraints"])
    gq, gv, _ = world.state()
    assert np.array_equal(gq.view(np.uint32), ost.q.view(np.uint32))
    assert np.array_equal(gv.view(np.uint32), ost.v.view(np.uint32))
