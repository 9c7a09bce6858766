"""The level schedule of the ordered sweeps against the oracle's plain index order, bit for bit, where
the schedule can go wrong: more than 64 levels (one slab under many boxes), more than 64 contacts
in few levels, an articulation touching dynamic bodies, one beside a dynamic body, and updates that are not finite (the first
failing contact in index order is reported)."""

import numpy as np
import pytest

import metalrobo as mr
import model_util as mu
import oracle_lib as ol

SPHERE, CAPSULE, BOX, PLANE = 0, 1, 2, 3


def box_inertia(m, h):
    return [m / 3.0 * (h[1] ** 2 + h[2] ** 2), m / 3.0 * (h[0] ** 2 + h[2] ** 2), m / 3.0 * (h[0] ** 2 + h[1] ** 2)]


def world(movers, links=(), dofs=(), link_shapes=(), nq=0, envs=2):
    """Dynamic boxes (half extents, mass) and spheres (radius, mass) over a plane, and optional links."""
    bodies = list(links) if links else [mu.body(1.0, [0.01] * 3)]
    nl = len(bodies)
    shapes = list(link_shapes)
    for dims, mass in movers:
        k = len(bodies)
        inertia = box_inertia(mass, dims) if len(dims) == 3 else [0.4 * mass * dims[0] ** 2] * 3
        bodies.append(mu.body(mass, inertia))
        shapes.append(mu.shape(k, BOX if len(dims) == 3 else SPHERE, dims))
    bodies.append(mu.body(0.0, [1, 1, 1], motion=0))
    shapes.append(mu.shape(len(bodies) - 1, PLANE, [], rot=mu.Y_TO_Z))
    return mu.CustomWorld(bodies, list(dofs), shapes, link_count=nl, root_type=0, nq=nq, nv=nq, envs=envs)


def beside(rng):
    """A chain of 20 box links lying on the plane and one free box apart: 80 levels of an articulated
    contact each, of which only the first four hold a contact between scene bodies too."""
    links, dofs, shapes = [mu.body(1.0, [0.01] * 3)], [], []
    for i in range(1, 21):
        links.append(mu.body(1.5, [0.02, 0.004, 0.02], parent=i - 1, joint_type=0, q_index=i - 1, v_index=i - 1,
                             axis=(0, 0, 1), parent_anchor=(0, 0.12, 0) if i > 1 else (0, 0, 0.0495),
                             child_anchor=(0, -0.12, 0)))
        dofs.append(mu.dof(i, i - 1))
        shapes.append(mu.shape(i, BOX, [0.1, 0.1, 0.05]))
    movers = [((0.06, 0.06, 0.06), 0.8)]
    w = world(movers, links, dofs, shapes, nq=20)
    return w, state_of(w, [(2.0, 0.0, 0.0595)], [0.8], rng), 20


def state_of(w, positions, masses, rng, speed=0.3):
    st = np.zeros((w.envs, len(masses) + 1), mr.BODY_STATE_DTYPE)
    for e in range(w.envs):
        for k, (p, m) in enumerate(zip(positions, masses)):
            st[e, k] = mu.scene_state(p, lin=rng.uniform(-speed, speed, 3), ang=rng.uniform(-1, 1, 3), inv_mass=1.0 / m)
        st[e, -1] = mu.scene_state((0, 0, 0), motion=0)
    return st


def slab(rng):
    """20 boxes on one slab: every contact touches the slab, so they form one chain of over 64 levels."""
    movers = [((0.6, 0.5, 0.05), 20.0)] + [((0.05, 0.05, 0.05), 0.5)] * 20
    positions = [(0, 0, 0.0495)] + [(-0.48 + 0.24 * (i % 5), -0.36 + 0.24 * (i // 5), 0.1485) for i in range(20)]
    w = world(movers)
    return w, state_of(w, positions, [m for _, m in movers], rng), 0


def grid(rng, heavy=()):
    """24 boxes and 20 spheres on the plane: over 64 contacts in a few wide levels."""
    movers = [((0.06, 0.05, 0.04), 50.0 if i in heavy else 0.7) for i in range(24)] + [((0.05,), 0.3)] * 20
    positions = [(0.115 * (i % 6), 0.14 * (i // 6), 0.0395) for i in range(24)]
    positions += [(0.095 * (i % 5) - 0.7, 0.099 * (i // 5), 0.049) for i in range(20)]
    w = world(movers)
    return w, state_of(w, positions, [m for _, m in movers], rng), 0


def linked(rng, heavy=(), apart=0):
    """Two capsule links lying on the plane among boxes: articulated contacts with dynamic endpoints;
    `apart` more boxes lie beside them."""
    links = [mu.body(1.0, [0.01] * 3)]
    dofs, shapes = [], []
    for i in (1, 2):
        links.append(mu.body(1.5, [0.02, 0.004, 0.02], parent=i - 1, joint_type=0, q_index=i - 1, v_index=i - 1,
                             axis=(0, 0, 1), parent_anchor=(0, 0.3, 0) if i > 1 else (0, 0, 0.0495),
                             child_anchor=(0, -0.3, 0)))
        dofs.append(mu.dof(i, i - 1))
        shapes.append(mu.shape(i, CAPSULE, [0.05, 0.2]))
    movers = [((0.06, 0.06, 0.06), 50.0 if i in heavy else 0.8) for i in range(8 + apart)]
    positions = [(0.109 if i % 2 else -0.109, 0.05 + 0.2 * (i // 2), 0.0595) for i in range(8)]
    positions += [(2.0 + i, 0.0, 0.0595) for i in range(apart)]
    w = world(movers, links, dofs, shapes, nq=2)
    return w, state_of(w, positions, [m for _, m in movers], rng), 2


def compare(w, scene, nq, steps=6, expect_failure=False, fails_at=None, **cfg_args):
    cfg = w.config(pair_capacity=256, manifold_capacity=128, constraint_capacity=256, **cfg_args)
    ost = ol.OracleState(w.model, cfg)
    gpu_world = mr.World(w.model, cfg)
    q = np.zeros((w.envs, nq), np.float32)
    ost.scene[:] = scene
    gpu_world.set_state(q, q, scene)
    cmd = np.zeros((w.envs, nq), np.float32)
    most = 0
    for k in range(steps):
        status, cs = ost.step(cmd, control_step=k)[:2]
        gpu_world.advance(cmd[None])
        got, gcs = gpu_world.statuses()[0], gpu_world.contact_statuses()[0]
        for f in ("code", "failing_index", "successful_substeps"):
            np.testing.assert_array_equal(got[f], status[f], err_msg=f"step {k} {f}")
        assert np.all((status["code"] != 0) == expect_failure)
        if fails_at is not None:
            # in a sweep: the oracle counts sweeps and takes residuals only after they all passed
            assert np.all(status["failing_index"] == fails_at), status["failing_index"]
            assert np.all(cs["solver_iterations"] == 0) and np.all(cs["constraints"] > fails_at)
            assert np.all(cs["residuals"] == 0.0)
        for f in ("constraints", "islands", "solver_iterations"):
            np.testing.assert_array_equal(gcs[f], cs[f], err_msg=f"step {k} {f}")
        np.testing.assert_array_equal(gcs["residuals"].view(np.uint32), cs["residuals"].view(np.uint32))
        gq, gv, gs = gpu_world.state()
        for a, b in ((gq, ost.q), (gv, ost.v), (gs, ost.scene)):
            assert np.array_equal(np.ascontiguousarray(a).view(np.uint8), np.ascontiguousarray(b).view(np.uint8)), k
        most = max(most, int(cs["constraints"].max()))
    return most


@pytest.mark.gpu
@pytest.mark.parametrize("tolerance", [0.0, 1.0e-5])
@pytest.mark.parametrize("scene,least", [(slab, 80), (grid, 65), (linked, 20), (beside, 84)])
def test_scheduled_sweeps_match_the_index_order(gpu, scene, least, tolerance):
    w, states, nq = scene(np.random.default_rng(4))
    assert compare(w, states, nq, residual_tolerance=tolerance) >= least


# An update is not finite where the impulse overflows: 50 kg stopped from 3e38 m/s. (The relative
# velocity itself is finite, so the evaluation before the sweeps passes.)
FAST = 3.0e38


@pytest.mark.gpu
def test_a_non_finite_update_reports_the_first_contact_in_index_order(gpu):
    """Box 5's contacts with the plane (40-43) lie at levels 20-23, behind its row's chain; box 6's
    (48-51) at levels 4-7: by level, 48 fails first."""
    for fast, fails_at in (((5, 6), 40), ((6,), 48)):
        for tolerance in (0.0, 1.0e-5):
            w, states, nq = grid(np.random.default_rng(4), heavy=(5, 6))
            for k in fast:
                states[:, k]["linear_velocity_inv_mass"][:, :3] = (0.0, 0.0, -FAST)
            compare(w, states, nq, steps=1, expect_failure=True, fails_at=fails_at, residual_tolerance=tolerance)


@pytest.mark.gpu
@pytest.mark.parametrize("tolerance", [0.0, 1.0e-5])
@pytest.mark.parametrize("fast,fails_at", [((6, 8), 8), ((6,), 8), ((8,), 44)])
def test_a_non_finite_articulated_update_reports_the_first_contact(gpu, fast, fails_at, tolerance):
    """Box 6 drives into a link (contact 8, behind the links' other contacts), box 8 lies apart: its
    contacts with the plane (44-47) lie at levels 0-3."""
    w, states, nq = linked(np.random.default_rng(4), heavy=(6, 8), apart=1)
    for k in fast:
        states[:, k]["linear_velocity_inv_mass"][:, :3] = (FAST, 0.0, 0.0) if k == 6 else (0.0, 0.0, -FAST)
    compare(w, states, nq, steps=1, expect_failure=True, fails_at=fails_at, residual_tolerance=tolerance)


@pytest.mark.gpu
def test_bodies_that_overflow_after_the_sweeps_report_the_first_one(gpu):
    w, states, nq = grid(np.random.default_rng(4))
    states = states.copy()
    # light enough for finite impulses; their motion overflows in the integration
    for k, e in ((40, 0), (9, 0), (30, 1), (31, 1)):
        w_bad = states[e, k]
        w_bad["linear_velocity_inv_mass"][:3] = (0.0, 0.0, -3.0e38)
        states[e, k] = w_bad
    compare(w, states, nq, steps=1, expect_failure=True)
