"""Muscle path geometry, activation -> torque operator and its gradient.

CPU tests pin the oracle against fp64 formulations that share no code with it (rotation
matrices, dense subtree masks instead of entry lists, the closed form of the reference's
own two-body fixture); GPU tests compare libimhip with the oracle bit for bit wherever only
IEEE-exact operations are involved and to 2e-6 where expf/cosf enter.
"""

import dataclasses
import gc

import numpy as np
import pytest
import torch

from instantmimic_amd import synth
from instantmimic_amd.muscle import warp_custom_ops as ops
from instantmimic_amd.muscle.muscle_dynamics import (
    MuscleDynamicsLayer,
    MuscleMechanics,
    MuscleTopology,
    build_dof_subtree_mask,
    build_muscle_sparse_torque_entries,
    build_torque_sparse_segment_entries,
    group_context_entries,
    group_context_rows,
    pack_context_entries,
)
from oracle import ref

FORCE_RTOL = 2e-6  # expf / cosf differ by a few ulp between libm and the GPU


# ---------------------------------------------------------------- fixtures


def fixture_layer(device="cpu", muscle_count=3, torque_dim=2, root_dof_count=6, mechanics=None):
    """The layer of the reference's tests/muscle_warp_fixtures.py:17-131: two bodies, one
    segment per muscle from (0,1,0) on the root body to (1,1,0) on the child."""
    nv = torque_dim + root_dof_count
    idx = np.arange(muscle_count)
    topo = MuscleTopology(
        muscle_params=np.tile(np.float32([[1.0, 1.0, 0.0, 0.0, 1.0]]), (muscle_count, 1)),
        muscle_rest_length=np.ones(muscle_count, np.float32),
        muscle_waypoints_local=np.tile(np.float32([[0, 1, 0], [1, 1, 0]]), (muscle_count, 1)),
        muscle_waypoint_body=np.tile([0, 1], muscle_count),
        all_segment_muscle_idx=idx, all_segment_start_idx=idx * 2, apply_segment_muscle_idx=idx,
        apply_segment_start_idx=idx * 2, apply_segment_end_idx=idx * 2 + 1,
        apply_segment_body_start_idx=np.zeros_like(idx), apply_segment_body_end_idx=np.ones_like(idx),
        body_parentid=np.array([0, 0]), body_rootid=np.array([0, 0]), dof_bodyid=np.array([0] * (nv - 1) + [1]),
    )  # fmt: skip
    mech = mechanics or MuscleMechanics(length_norm_min=0.2, length_norm_max=1.4)
    return MuscleDynamicsLayer(topo, body_count=2, full_torque_dim=nv, torque_dim=torque_dim,
                               muscle_count=muscle_count, mechanics=mech, device=device)  # fmt: skip


def fixture_context(layer, batch=4):
    """tests/muscle_warp_fixtures.py:151-180: child body at x = 1, identity orientations,
    the last torque dof rotates about z."""
    body = np.zeros((batch, layer.body_count, 3), np.float32)
    body[:, 1, 0] = 1.0
    quat = np.zeros((batch, layer.body_count, 4), np.float32)
    quat[..., 0] = 1.0
    cdof = np.zeros((batch, layer.full_torque_dim, 6), np.float32)
    cdof[:, layer.root_dof_count + layer.torque_dim - 1, 2] = 1.0
    flat = [a.reshape(batch, int(np.prod(a.shape[1:]))) for a in (body, quat, body, body, cdof)]
    return np.concatenate(flat, axis=1)


def split_context(layer, ctx):
    nb, nv = layer.body_count, layer.full_torque_dim
    B = ctx.shape[0]
    xpos = ctx[:, : 3 * nb].reshape(B, nb, 3)
    xquat = ctx[:, 3 * nb : 7 * nb].reshape(B, nb, 4)
    com = ctx[:, 10 * nb : 13 * nb].reshape(B, nb, 3)
    cdof = ctx[:, 13 * nb : 13 * nb + 6 * nv].reshape(B, nv, 6)
    return xpos, xquat, com, cdof


def model9(mech: MuscleMechanics):
    return np.float32([mech.force_scale, mech.length_norm_min, mech.length_norm_max, *mech.active_params(),
                       *mech.passive_params()])  # fmt: skip


def oracle_forward(layer, ctx, act, include_passive, unit=None, passive=None, waypoints=None):
    xpos, xquat, com, cdof = split_context(layer, ctx)
    wp = ref.muscle_waypoints(xpos, xquat, layer.waypoint_body, layer.waypoints_local) if waypoints is None else waypoints
    if unit is None:
        unit, passive = ref.muscle_force_magnitudes(
            wp, layer.all_segment_start_idx, layer.all_muscle_segment_offsets, layer.muscle_params,
            layer.muscle_rest_length, model9(layer.mechanics), include_passive,
        )  # fmt: skip
    tq = layer.torque_entries_host
    out = ref.muscle_torque_forward(
        wp, com, cdof, layer.segments_host, (tq[0], tq[2], tq[3], tq[4], tq[5]), unit,
        passive if include_passive else None, act, layer.root_dof_count,
    )  # fmt: skip
    return out, wp, unit, passive


def oracle_backward(layer, ctx, gout, wp, unit):
    _, _, com, cdof = split_context(layer, ctx)
    return ref.muscle_activation_grad(wp, com, cdof, layer.segments_host, layer.muscle_entries_host, unit, gout,
                                      layer.root_dof_count)  # fmt: skip


# ---------------------------------------------------------------- fp64 references (independent)


def rotmat64(q):
    q = q.astype(np.float64)
    q = q / np.sqrt((q * q).sum(-1, keepdims=True) + 1e-8)
    w, x, y, z = np.moveaxis(q, -1, 0)
    return np.stack(
        [1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
         2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
         2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], axis=-1,
    ).reshape(q.shape[:-1] + (3, 3))  # fmt: skip


def waypoints64(layer, xpos, xquat):
    R = rotmat64(xquat)[:, layer.waypoint_body]
    return xpos.astype(np.float64)[:, layer.waypoint_body] + np.einsum("bwij,wj->bwi", R, layer.waypoints_local.astype(np.float64))


def curves64(mech, ln):
    if mech.active_force_type == "gaussian":
        fa = np.exp(-((ln - 1) ** 2) / mech.active_force_gamma)
    else:
        lmin, lmax = mech.active_force_lmin, mech.active_force_lmax
        lo, hi = 0.5 * (lmin + 1), 0.5 * (1 + lmax)
        fa = np.select(
            [(ln < lmin) | (ln > lmax), ln <= lo, ln <= 1.0, ln <= hi],
            [0.0, 0.5 * ((ln - lmin) / (lo - lmin)) ** 2, 1 - 0.5 * ((1 - ln) / (1 - lo)) ** 2,
             1 - 0.5 * ((ln - 1) / (hi - 1)) ** 2],
            0.5 * ((lmax - ln) / (lmax - hi)) ** 2,
        )  # fmt: skip
    if mech.passive_force_type == "exponential":
        k, e = mech.passive_force_k_pe, mech.passive_force_e_mo
        fp = np.where(ln < 1, 0.0, (np.exp(np.clip(k * (ln - 1) / e, -80, 80)) - 1) / (np.exp(k) - 1))
    else:
        lmax, fpmax = mech.passive_force_lmax, mech.passive_force_fpmax
        mid = 0.5 * (1 + lmax)
        w = mid - 1
        fp = np.select([ln <= 1, ln <= mid], [0.0, 0.5 * fpmax * ((ln - 1) / w) ** 2], fpmax * (0.5 + (ln - mid) / w))
    return fa, fp


def forces64(layer, wp):
    mech = layer.mechanics
    seg_len = np.linalg.norm(wp[:, layer.all_segment_start_idx + 1] - wp[:, layer.all_segment_start_idx], axis=-1)
    length = np.zeros((wp.shape[0], layer.muscle_count))
    muscle_of = np.repeat(np.arange(layer.muscle_count), np.diff(layer.all_muscle_segment_offsets))
    np.add.at(length, (slice(None), muscle_of), seg_len)
    p = layer.muscle_params.astype(np.float64)
    ln = np.clip((length / np.maximum(layer.muscle_rest_length, 1e-6) - p[:, 2]) / np.maximum(p[:, 1], 1e-6),
                 np.float32(mech.length_norm_min), np.float32(mech.length_norm_max))  # fmt: skip
    fa, fp = curves64(mech, ln)
    gain = p[:, 0] * np.cos(p[:, 3]) * mech.force_scale
    return gain * fa, gain * fp, ln


def moment_matrix64(layer, wp, com, cdof):
    """T[b, j, m] = d torque_j / d force_m from the dense subtree masks."""
    p0i, p1i, b0, b1 = layer.segments_host
    com = com.astype(np.float64)
    cd = cdof.astype(np.float64)[:, layer.root_dof_count :]
    ang, lin = cd[..., :3], cd[..., 3:]
    p0, p1 = wp[:, p0i], wp[:, p1i]
    seg = p1 - p0
    length = np.linalg.norm(seg, axis=-1, keepdims=True)
    u = np.where(length < 1e-8, 0.0, seg / np.maximum(length, 1e-300))
    r0, r1 = p0 - com[:, b0], p1 - com[:, b1]
    # (lin + ang x r) . u = lin . u + ang . (r x u)
    t0 = np.einsum("bjc,bsc->bjs", lin, u) + np.einsum("bjc,bsc->bjs", ang, np.cross(r0, u))
    t1 = np.einsum("bjc,bsc->bjs", lin, u) + np.einsum("bjc,bsc->bjs", ang, np.cross(r1, u))
    per_seg = layer.segment_start_dof_mask[None] * t0 - layer.segment_end_dof_mask[None] * t1
    onehot = np.zeros((len(p0i), layer.muscle_count))
    onehot[np.arange(len(p0i)), layer.apply_segment_muscle_idx] = 1.0
    return per_seg @ onehot


@pytest.fixture(scope="module")
def rig_layer():
    rig = synth.make_muscle_rig(nmuscle=60, seed=5)
    mech = MuscleMechanics(length_norm_min=0.2, length_norm_max=1.8)
    return rig, MuscleDynamicsLayer(rig.topology, **rig.dims(), mechanics=mech, device="cpu")


# ---------------------------------------------------------------- host tables


def test_subtree_mask_and_entry_tables():
    parent = [0, 0, 1, 2, 1]
    dof_body = [0, 0, 1, 2, 2, 3, 4]
    mask = build_dof_subtree_mask(parent, dof_body, 5, 7)
    # brute force: dof on body d moves body b when d is b or an ancestor of b; world dofs move all
    for d, db in enumerate(dof_body):
        for b in range(5):
            chain, p = [], b
            while p != 0:
                chain.append(p)
                p = parent[p]
            assert mask[d, b] == (1.0 if db == 0 or db in chain else 0.0)
    rng = np.random.default_rng(3)
    start = (rng.random((5, 9)) < 0.4).astype(np.float32)
    end = (rng.random((5, 9)) < 0.4).astype(np.float32)
    muscle = rng.integers(0, 4, 9)
    off, tq, seg, mus, a, b = build_torque_sparse_segment_entries(start, end, muscle)
    want = [(j, s) for j in range(5) for s in range(9) if start[j, s] or end[j, s]]
    assert list(zip(tq.tolist(), seg.tolist())) == want
    assert off.tolist() == [sum(1 for j, _ in want if j < k) for k in range(6)]
    assert np.array_equal(mus, muscle[seg]) and np.array_equal(a, start[tq, seg]) and np.array_equal(b, end[tq, seg])
    moff, mseg, mtq, ma, mb = build_muscle_sparse_torque_entries(off, seg, a, b, muscle, 4)
    keys = [(int(muscle[s]), int(s), int(j)) for s, j in zip(mseg, mtq)]
    assert keys == sorted((int(muscle[s]), s, j) for j, s in want)
    assert moff.tolist() == [sum(1 for k in keys if k[0] < m) for m in range(5)]
    assert np.array_equal(ma, start[mtq, mseg]) and np.array_equal(mb, end[mtq, mseg])


def test_layer_validates_its_inputs():
    with pytest.raises(ValueError):
        MuscleMechanics(active_force_type="cubic")
    with pytest.raises(ValueError):
        MuscleMechanics(active_force_lmin=1.2)
    with pytest.raises(NotImplementedError):
        MuscleMechanics(force_velocity_enabled=True)
    layer = fixture_layer()
    with pytest.raises(RuntimeError, match="no CPU path"):
        layer._warp_muscle_dynamics_from_activation_forward(
            torch.zeros(4, 3), torch.from_numpy(fixture_context(layer)), include_passive_force=False
        )


# ---------------------------------------------------------------- oracle pinning


def test_oracle_waypoints_against_rotation_matrices(rig_layer):
    rig, layer = rig_layer
    ctx = synth.make_muscle_context(rig, 16, seed=2)
    xpos, xquat, _, _ = split_context(layer, ctx)
    got = ref.muscle_waypoints(xpos, xquat, layer.waypoint_body, layer.waypoints_local)
    want = waypoints64(layer, xpos, xquat)
    assert np.abs(got - want).max() < 2e-6
    # identity orientation: a pure translation, exactly
    q = np.zeros_like(xquat)
    q[..., 0] = 1.0
    got = ref.muscle_waypoints(xpos, q, layer.waypoint_body, layer.waypoints_local)
    assert np.abs(got - (xpos[:, layer.waypoint_body] + layer.waypoints_local)).max() < 1e-7


@pytest.mark.parametrize("active", ["gaussian", "mujoco"])
@pytest.mark.parametrize("passive", ["exponential", "mujoco"])
def test_oracle_force_magnitudes_against_fp64_curves(active, passive):
    rig = synth.make_muscle_rig(nmuscle=60, seed=5)
    mech = MuscleMechanics(active_force_type=active, passive_force_type=passive, length_norm_min=0.2, length_norm_max=1.8)
    layer = MuscleDynamicsLayer(rig.topology, **rig.dims(), mechanics=mech, device="cpu")
    ctx = synth.make_muscle_context(rig, 32, seed=4)
    ctx[:, : 3 * rig.body_count] *= 0.5  # spread the normalised lengths over every branch of the curves
    xpos, xquat, _, _ = split_context(layer, ctx)
    wp = ref.muscle_waypoints(xpos, xquat, layer.waypoint_body, layer.waypoints_local)
    unit, pas = ref.muscle_force_magnitudes(wp, layer.all_segment_start_idx, layer.all_muscle_segment_offsets,
                                            layer.muscle_params, layer.muscle_rest_length, model9(mech), True)  # fmt: skip
    u64, p64, ln = forces64(layer, wp.astype(np.float64))
    assert (ln < 1).any() and (ln > 1.3).any() and ((ln > 1) & (ln < 1.3)).any()
    scale = layer.muscle_params[:, 0].max()
    assert np.abs(unit - u64).max() < 2e-5 * scale
    assert np.abs(pas - p64).max() < 2e-5 * max(scale, np.abs(p64).max())
    _, zero = ref.muscle_force_magnitudes(wp, layer.all_segment_start_idx, layer.all_muscle_segment_offsets,
                                          layer.muscle_params, layer.muscle_rest_length, model9(mech), False)  # fmt: skip
    assert not zero.any()


def test_oracle_on_the_reference_fixture_closed_form():
    layer = fixture_layer()
    ctx = fixture_context(layer)
    act = np.float32([[0.1, 0.5, 0.9]] * 4)
    out, wp, unit, _ = oracle_forward(layer, ctx, act, False)
    # waypoints (0,1,0) and (2,1,0): length 2, normalised length clamped to 1.4
    assert np.array_equal(wp[0].reshape(-1, 3)[:2], np.float32([[0, 1, 0], [2, 1, 0]]))
    u = np.exp(-(0.4**2) / 0.45)
    assert np.allclose(unit, u, rtol=1e-6)
    # only the child's z rotation sees the muscles: lever (2,1,0), pull along x => torque = +F
    assert np.all(out[:, 0] == 0)
    assert np.allclose(out[:, 1], u * act.sum(1), rtol=1e-6)
    grad = oracle_backward(layer, ctx, np.float32([[0.0, 2.0]] * 4), wp, unit)
    assert np.allclose(grad, 2.0 * u, rtol=1e-6)


def test_oracle_contractions_against_dense_fp64(rig_layer):
    rig, layer = rig_layer
    B = 8
    ctx = synth.make_muscle_context(rig, B, seed=7)
    rng = np.random.default_rng(11)
    act = rng.uniform(0, 1, (B, rig.muscle_count)).astype(np.float32)
    act[:, ::7] = 0.0  # exercises the force == 0 skip
    out, wp, unit, pas = oracle_forward(layer, ctx, act, True)
    _, _, com, cdof = split_context(layer, ctx)
    T = moment_matrix64(layer, wp.astype(np.float64), com, cdof)  # (B, torque, muscle)
    force = unit.astype(np.float64) * act + pas
    want = np.einsum("bjm,bm->bj", T, force)
    assert ref.rel_l2(out, want) < 2e-6
    no_passive, *_ = oracle_forward(layer, ctx, act, False)
    assert ref.rel_l2(no_passive, np.einsum("bjm,bm->bj", T, unit.astype(np.float64) * act)) < 2e-6
    # gradient = transpose of the same linear map, scaled by the unit force
    g = rng.normal(0, 1, (B, rig.torque_dim)).astype(np.float32)
    grad = oracle_backward(layer, ctx, g, wp, unit)
    assert ref.rel_l2(grad, np.einsum("bjm,bj->bm", T, g.astype(np.float64)) * unit) < 2e-6
    # sparse moment: the nonzero pattern of T, entry by entry
    e = layer.sparse_entries
    mom = ref.muscle_sparse_moment(wp, com, cdof, layer.segments_host, e.muscle_dof_torque_idx,
                                   e.muscle_dof_segment_offsets, e.segment_idx, e.start_coeff, e.end_coeff,
                                   layer.root_dof_count)  # fmt: skip
    assert ref.rel_l2(mom, T[:, e.muscle_dof_torque_idx, e.muscle_dof_muscle_idx]) < 2e-6
    dense = np.zeros_like(T)
    dense[:, e.muscle_dof_torque_idx, e.muscle_dof_muscle_idx] = mom
    assert np.abs(dense - T).max() < 1e-5 * np.abs(T).max()  # nothing of T lies off the entry list


def test_oracle_bounds_against_dense_fp64(rig_layer):
    rig, layer = rig_layer
    ctx = synth.make_muscle_context(rig, 8, seed=17)
    _, wp, unit, _ = oracle_forward(layer, ctx, np.ones((8, rig.muscle_count), np.float32), False)
    _, _, com, cdof = split_context(layer, ctx)
    tq = layer.torque_entries_host
    lo, hi = ref.muscle_torque_bounds(wp, com, cdof, layer.segments_host, (tq[0], tq[2], tq[3], tq[4], tq[5]), unit,
                                      layer.root_dof_count)  # fmt: skip
    per_muscle = moment_matrix64(layer, wp.astype(np.float64), com, cdof) * unit[:, None, :]
    assert ref.rel_l2(lo, np.minimum(per_muscle, 0).sum(-1)) < 2e-6
    assert ref.rel_l2(hi, np.maximum(per_muscle, 0).sum(-1)) < 2e-6
    assert (lo <= 0).all() and (hi >= 0).all()


def test_oracle_degenerate_segment_contributes_nothing():
    layer = fixture_layer()
    ctx = fixture_context(layer)
    ctx[:, 3] = -1.0  # child body at x = -1: both waypoints coincide at (0,1,0)
    out, wp, unit, _ = oracle_forward(layer, ctx, np.ones((4, 3), np.float32), False)
    assert np.array_equal(wp[0].reshape(-1, 3)[0], wp[0].reshape(-1, 3)[1])
    assert not out.any()


# ---------------------------------------------------------------- operator registry (no GPU)


def test_operator_schemas_and_registry():
    fwd = torch.ops.instantmimic_muscle.torque_forward.default
    bwd = torch.ops.instantmimic_muscle.torque_backward.default
    assert str(fwd._schema) == (
        "instantmimic_muscle::torque_forward(Tensor activation, Tensor raw_context, SymInt layer_key, "
        "bool include_passive_force) -> Tensor"
    )
    assert str(bwd._schema) == (
        "instantmimic_muscle::torque_backward(Tensor raw_context, Tensor grad_output, SymInt layer_key) -> Tensor"
    )
    layer = fixture_layer()
    key = ops.warp_op_key(layer)
    assert ops.warp_op_key(layer) == key and ops._layer_for(key) is layer
    import copy

    clone = copy.copy(layer)
    assert clone._warp_op_key == key and ops.warp_op_key(clone) != key  # a copy gets its own handle
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode():
        a = torch.empty(5, 3)
        c = torch.empty(5, layer.context_dim)
        assert ops.muscle_torque_forward(a, c, key, False).shape == (5, 2)
        assert ops.muscle_torque_backward(c, torch.empty(5, 2), key).shape == (5, 3)
        u = torch.empty(5, 3)
        assert ops.muscle_torque_cached_lbs_forward(a, c, u, u, key, True).shape == (5, 2)
        assert ops.muscle_torque_cached_lbs_backward(c, u, torch.empty(5, 2), key).shape == (5, 3)
        lo, hi = ops.muscle_torque_bounds(c, key, True)
        assert lo.shape == hi.shape == (5, 2)
    del layer
    gc.collect()
    with pytest.raises(RuntimeError, match="not registered"):
        ops._layer_for(key)


# ---------------------------------------------------------------- GPU parity


def _gpu_layer(rig, **mech):
    m = MuscleMechanics(length_norm_min=0.2, length_norm_max=1.8, **mech)
    return MuscleDynamicsLayer(rig.topology, **rig.dims(), mechanics=m, device="cuda")


@pytest.mark.gpu
@pytest.mark.parametrize("active,passive", [("gaussian", "exponential"), ("mujoco", "mujoco")])
@pytest.mark.parametrize("nworld", [1, 67, 1024])
def test_gpu_geometry_forward_backward_match_oracle(active, passive, nworld):
    rig = synth.make_muscle_rig(nmuscle=284, seed=1003)
    layer = _gpu_layer(rig, active_force_type=active, passive_force_type=passive)
    ctx = synth.make_muscle_context(rig, nworld, seed=9)
    ctx[:, : 3 * rig.body_count] *= 0.5
    rng = np.random.default_rng(13)
    act = rng.uniform(0, 1, (nworld, rig.muscle_count)).astype(np.float32)
    act[:, ::5] = 0.0
    g = rng.normal(0, 1, (nworld, rig.torque_dim)).astype(np.float32)
    ctx_d, act_d = torch.from_numpy(ctx).cuda(), torch.from_numpy(act).cuda()
    for include_passive in (False, True):
        mean, wp_d, unit_d = layer._warp_muscle_dynamics_from_activation_forward(
            act_d, ctx_d, include_passive_force=include_passive
        )
        ws, _ = layer._prepare_waypoint_geometry(ctx_d, include_passive_force_magnitude=include_passive)
        torch.cuda.synchronize()
        wp = wp_d.cpu().numpy().reshape(nworld, -1, 3)
        unit, pas = unit_d.cpu().numpy(), ws["passive_force_magnitude"].cpu().numpy()
        want, wp_o, unit_o, pas_o = oracle_forward(layer, ctx, act, include_passive)
        assert np.array_equal(wp, wp_o)  # IEEE-exact operations only
        scale = np.abs(unit_o).max()
        assert np.abs(unit - unit_o).max() <= FORCE_RTOL * scale
        assert np.abs(pas - pas_o).max() <= FORCE_RTOL * max(scale, np.abs(pas_o).max())
        if not include_passive:
            assert not pas.any()
        # the contraction itself, from the GPU's own force magnitudes: bit exact
        exact, *_ = oracle_forward(layer, ctx, act, include_passive, unit=unit, passive=pas, waypoints=wp)
        assert np.array_equal(mean.cpu().numpy(), exact)
        assert ref.rel_l2(mean.cpu().numpy(), want) < 1e-5
    grad = layer._warp_muscle_dynamics_from_activation_backward(ctx_d, torch.from_numpy(g).cuda())
    assert np.array_equal(grad.cpu().numpy(), oracle_backward(layer, ctx, g, wp, unit))
    cached = layer._warp_muscle_dynamics_from_activation_backward(ctx_d, torch.from_numpy(g).cuda(), unit_d)
    assert torch.equal(cached, grad)


@pytest.mark.gpu
def test_gpu_sparse_moment_matches_oracle_and_feeds_the_projection():
    from instantmimic_amd.muscle import muscle_qfrc_projector as proj

    rig = synth.make_muscle_rig(nmuscle=284, seed=1003)
    layer = _gpu_layer(rig)
    nworld = 257
    ctx = synth.make_muscle_context(rig, nworld, seed=21)
    ctx_d = torch.from_numpy(ctx).cuda()
    mom = layer.eval_muscle_sparse_moment(ctx_d)
    ws, _ = layer._prepare_waypoint_geometry(ctx_d, include_passive_force_magnitude=False)
    wp = ws["transformed_waypoints"].cpu().numpy().reshape(nworld, -1, 3)
    _, _, com, cdof = split_context(layer, ctx)
    e = layer.sparse_entries
    want = ref.muscle_sparse_moment(wp, com, cdof, layer.segments_host, e.muscle_dof_torque_idx,
                                    e.muscle_dof_segment_offsets, e.segment_idx, e.start_coeff, e.end_coeff,
                                    layer.root_dof_count)  # fmt: skip
    assert np.array_equal(mom.cpu().numpy(), want)
    # tau = A' f through the projection kernel equals the operator's torque to rounding
    act = torch.rand(nworld, rig.muscle_count, device="cuda")
    force = ws["unit_force_magnitude"] * act
    offsets, entry_idx = proj.torque_sorted_entries(e.muscle_dof_torque_idx, rig.torque_dim)
    qfrc = torch.zeros(nworld, rig.full_torque_dim, device="cuda")
    proj.project_muscle_sparse_moment_qfrc(
        mom, force, torch.from_numpy(offsets).cuda(), torch.from_numpy(entry_idx).cuda(),
        torch.from_numpy(e.muscle_dof_muscle_idx.astype(np.int32)).cuda(), layer.root_dof_count, qfrc,
    )  # fmt: skip
    torque = layer.forward_from_activation(act, ctx_d, False)
    assert ref.rel_l2(qfrc[:, layer.root_dof_count :].cpu().numpy(), torque.cpu().numpy()) < 1e-5
    assert not qfrc[:, : layer.root_dof_count].any()


@pytest.mark.gpu
def test_gpu_operator_fixture_closed_form_autograd_and_compile():
    layer = fixture_layer("cuda")
    ctx = torch.from_numpy(fixture_context(layer)).cuda()
    key = ops.warp_op_key(layer)
    u = float(np.exp(-(0.4**2) / 0.45))

    def loss(a):
        return ops.muscle_torque_forward(a.sin(), ctx, key, False).square().sum()

    a = torch.full((4, 3), 0.4, device="cuda", requires_grad=True)
    value = loss(a)
    (grad,) = torch.autograd.grad(value, a)
    s, c = np.sin(0.4), np.cos(0.4)
    assert abs(value.item() - 4 * (3 * u * s) ** 2) < 1e-5 * value.item()
    assert torch.allclose(grad, torch.full_like(grad, 2 * (3 * u * s) * u * c), rtol=1e-5)
    assert torch.count_nonzero(grad) > 0
    # strict fullgraph compilation reaches the kernels only through the dispatcher operators
    compiled = torch.compile(loss, fullgraph=True, backend="aot_eager")
    b = torch.full((4, 3), 0.4, device="cuda", requires_grad=True)
    cvalue = compiled(b)
    (cgrad,) = torch.autograd.grad(cvalue, b)
    assert torch.equal(cvalue, value) and torch.equal(cgrad, grad)
    # the autograd node keeps the layer alive after the caller dropped it
    pending = loss(torch.full((4, 3), 0.2, device="cuda", requires_grad=True))
    del layer
    gc.collect()
    pending.backward()


@pytest.mark.gpu
def test_gpu_cached_force_ops_and_bounds():
    rig = synth.make_muscle_rig(nmuscle=284, seed=1003)
    active = np.arange(0, rig.torque_dim, 3)
    layer = MuscleDynamicsLayer(rig.topology, **rig.dims(), mechanics=MuscleMechanics(), active_torque_indices=active,
                                device="cuda")  # fmt: skip
    nworld = 93
    ctx = synth.make_muscle_context(rig, nworld, seed=31)
    ctx_d = torch.from_numpy(ctx).cuda()
    key = ops.warp_op_key(layer)
    act = torch.rand(nworld, rig.muscle_count, device="cuda", requires_grad=True)
    torque = ops.muscle_torque_forward(act, ctx_d, key, True)
    ws, _ = layer._prepare_waypoint_geometry(ctx_d, include_passive_force_magnitude=True)
    unit, pas = ws["unit_force_magnitude"], ws["passive_force_magnitude"]
    cached = ops.muscle_torque_cached_lbs_forward(act, ctx_d, unit, pas, key, True)
    assert torch.equal(cached, torque)
    g = torch.randn_like(torque)
    (g1,) = torch.autograd.grad(torque, act, g, retain_graph=True)
    (g2,) = torch.autograd.grad(cached, act, g)
    assert torch.equal(g1, g2) and torch.count_nonzero(g1) > 0
    lo, hi = ops.muscle_torque_bounds(ctx_d, key, False)
    wp = ws["transformed_waypoints"].cpu().numpy().reshape(nworld, -1, 3)
    _, _, com, cdof = split_context(layer, ctx)
    tq = layer.torque_entries_host
    want_lo, want_hi = ref.muscle_torque_bounds(wp, com, cdof, layer.segments_host,
                                                (tq[0], tq[2], tq[3], tq[4], tq[5]), unit.cpu().numpy(),
                                                layer.root_dof_count)  # fmt: skip
    assert np.array_equal(lo.cpu().numpy(), want_lo) and np.array_equal(hi.cpu().numpy(), want_hi)
    # activations in [0, 1] without passive force stay inside the box
    inside = ops.muscle_torque_forward(act.detach(), ctx_d, key, False)
    tol = 1e-4 * hi.abs().max()
    assert (inside >= lo - tol).all() and (inside <= hi + tol).all()
    slo, shi = ops.muscle_torque_bounds(ctx_d, key, True)
    assert torch.equal(slo, lo[:, active]) and torch.equal(shi, hi[:, active])


@pytest.mark.gpu
def test_gpu_edge_cases():
    layer = fixture_layer("cuda")
    ctx = torch.from_numpy(fixture_context(layer, batch=0)).cuda()
    out, _, _ = layer._warp_muscle_dynamics_from_activation_forward(
        torch.zeros(0, 3, device="cuda"), ctx, include_passive_force=True
    )
    assert out.shape == (0, 2)
    # a context that carries trailing columns (strided rows) and degenerate segments
    full = fixture_context(layer, batch=5)
    full[:, 3] = -1.0
    wide = torch.zeros(5, layer.context_dim + 9, device="cuda")
    wide[:, : layer.context_dim] = torch.from_numpy(full).cuda()
    out, _, _ = layer._warp_muscle_dynamics_from_activation_forward(
        torch.ones(5, 3, device="cuda"), wide[:, : layer.context_dim + 3], include_passive_force=False
    )
    assert not out.any()
    with pytest.raises(ValueError):
        layer._warp_muscle_dynamics_from_activation_forward(
            torch.ones(5, 2, device="cuda"), wide, include_passive_force=False
        )
    with pytest.raises(ValueError, match="columns"):
        layer._warp_muscle_dynamics_from_activation_forward(
            torch.ones(5, 3, device="cuda"), wide[:, :20].contiguous(), include_passive_force=False
        )


@pytest.mark.gpu
def test_gpu_one_thread_per_output_kernels_agree():
    """The contractions have two kernels each (a workgroup per world with the segments staged in
    LDS, and one thread per output for models that do not fit): the second one is forced here
    in a child process and must pass the same oracle comparison."""
    import os
    import subprocess
    import sys

    env = dict(os.environ, IMHIP_MUSCLE_KERNEL="simple")
    code = (
        "import sys; sys.path.insert(0, 'tests'); import test_muscle_dynamics as t;"
        "t.test_gpu_geometry_forward_backward_match_oracle('gaussian', 'exponential', 67);"
        "t.test_gpu_sparse_moment_matches_oracle_and_feeds_the_projection();"
        "t.test_gpu_cached_force_ops_and_bounds(); print('simple kernels ok')"
    )
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", code], cwd=root, env=env, capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and "simple kernels ok" in out.stdout, out.stderr[-2000:]


@pytest.mark.gpu
@pytest.mark.parametrize("nworld", [1, 333])
def test_gpu_fused_geometry_equals_the_two_launches(nworld):
    """im_muscle_waypoints_forces against im_muscle_waypoints followed by
    im_muscle_force_magnitudes, through the C-ABI: the same bits, rows beyond the outputs'
    widths untouched."""
    import ctypes as C

    from instantmimic_amd import _lib

    rig = synth.make_muscle_rig(nmuscle=284, seed=1003)
    layer = _gpu_layer(rig, active_force_type="gaussian", passive_force_type="exponential")
    ctx_d = torch.from_numpy(synth.make_muscle_context(rig, nworld, seed=21)).cuda()
    ws, _ = layer._prepare_waypoint_geometry(ctx_d, include_passive_force_magnitude=True)
    d, L = layer._dev, _lib.lib()
    base, ld = ctx_d.data_ptr(), ctx_d.stride(0)
    pad = 5
    wp = torch.full((nworld, 3 * layer.waypoint_count + pad), 7.0, device="cuda")
    unit = torch.full((nworld, layer.muscle_count + pad), 7.0, device="cuda")
    pas = torch.full((nworld, layer.muscle_count + pad), 7.0, device="cuda")
    wp_args = (base + 4 * layer._xpos_off, ld, base + 4 * layer._xquat_off, ld, d["wp_body"].data_ptr(),
               d["wp_local"].data_ptr(), layer.waypoint_count, wp.data_ptr(), wp.stride(0))  # fmt: skip
    frc_args = (d["all_seg_start"].data_ptr(), d["all_seg_off"].data_ptr(), d["params"].data_ptr(),
                layer.muscle_params.shape[1], d["rest"].data_ptr(), C.byref(layer._model), layer.muscle_count,
                unit.data_ptr(), unit.stride(0), pas.data_ptr(), pas.stride(0), nworld, None)  # fmt: skip
    _lib.check(L.im_muscle_waypoints(*wp_args, nworld, None), "im_muscle_waypoints")
    _lib.check(L.im_muscle_force_magnitudes(wp.data_ptr(), wp.stride(0), *frc_args), "im_muscle_force_magnitudes")
    torch.cuda.synchronize()
    assert torch.equal(wp[:, :-pad], ws["transformed_waypoints"])
    assert torch.equal(unit[:, :-pad], ws["unit_force_magnitude"])
    assert torch.equal(pas[:, :-pad], ws["passive_force_magnitude"])
    assert (wp[:, -pad:] == 7.0).all() and (unit[:, -pad:] == 7.0).all() and (pas[:, -pad:] == 7.0).all()
    # the fused call with padded rows as well
    wp2, unit2, pas2 = torch.full_like(wp, 3.0), torch.full_like(unit, 3.0), torch.full_like(pas, 3.0)
    args2 = wp_args[:7] + (wp2.data_ptr(), wp2.stride(0)) + frc_args[:7] + (
        unit2.data_ptr(), unit2.stride(0), pas2.data_ptr(), pas2.stride(0), nworld, None)  # fmt: skip
    _lib.check(L.im_muscle_waypoints_forces(*args2), "im_muscle_waypoints_forces")
    torch.cuda.synchronize()
    assert torch.equal(wp2[:, :-pad], wp[:, :-pad]) and torch.equal(unit2[:, :-pad], unit[:, :-pad])
    assert torch.equal(pas2[:, :-pad], pas[:, :-pad])
    assert (wp2[:, -pad:] == 3.0).all() and (unit2[:, -pad:] == 3.0).all() and (pas2[:, -pad:] == 3.0).all()


@pytest.mark.gpu
def test_gpu_entry_lists_without_a_stated_range_take_the_other_kernels():
    """An entry list whose nother field is 0 sends the contractions to the one-thread-per-output
    kernels; results are the same bits as with the range stated."""
    rig = synth.make_muscle_rig(nmuscle=284, seed=1003)
    layer = _gpu_layer(rig, active_force_type="gaussian", passive_force_type="exponential")
    nworld = 77
    ctx_d = torch.from_numpy(synth.make_muscle_context(rig, nworld, seed=5)).cuda()
    act = torch.rand(nworld, rig.muscle_count, device="cuda")
    g = torch.randn(nworld, rig.torque_dim, device="cuda")

    def run():
        mean, _, unit = layer._warp_muscle_dynamics_from_activation_forward(act, ctx_d, include_passive_force=True)
        grad = layer._warp_muscle_dynamics_from_activation_backward(ctx_d, g)
        moment = layer.eval_muscle_sparse_moment(ctx_d)
        torch.cuda.synchronize()
        return mean.clone(), grad.clone(), moment.clone()

    stated = run()
    for e in (layer._torque_entries, layer._muscle_entries, layer._moment_entries):
        assert e.nother > 0
        e.nother = 0
    for a, b in zip(stated, run()):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("muscles", [8, 96, 104, 210, 284, 340])
def test_gpu_contractions_of_many_worlds_equal_one_world_per_workgroup(muscles):
    """More worlds than workgroups (a workgroup then takes several, with a remainder), rigs on both
    sides of the entries a thread keeps (two, four, six; more are read per world): the bits of the
    one-thread-per-output kernels."""
    rig = synth.make_muscle_rig(nmuscle=muscles, seed=1003)
    layer = _gpu_layer(rig)
    nworld = 1100
    ctx_d = torch.from_numpy(synth.make_muscle_context(rig, nworld, seed=6)).cuda()
    act = torch.rand(nworld, rig.muscle_count, device="cuda")
    act[:, ::7] = 0.0
    g = torch.randn(nworld, rig.torque_dim, device="cuda")

    def run():
        mean, _, unit = layer._warp_muscle_dynamics_from_activation_forward(act, ctx_d, include_passive_force=False)
        lo, hi = layer._compute_activation_torque_bounds_warp(ctx_d, select_active=False)
        return mean, layer._warp_muscle_dynamics_from_activation_backward(ctx_d, g), layer.eval_muscle_sparse_moment(ctx_d), lo, hi

    kept = run()
    for e in (layer._torque_entries, layer._muscle_entries, layer._moment_entries):
        e.nother = 0
    for a, b in zip(kept, run()):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("muscles", [29, 30, 63, 64, 94, 95, 131, 132])
def test_gpu_contractions_on_every_workgroup_size(muscles):
    """Both sides of 512, 1024, 1536 and 2048 entries, where a workgroup's threads and the entries they
    keep change, in batches below and above those in which workgroups keep any (1536 and 3584 worlds):
    the bits of the one-thread-per-output kernels."""
    rig = synth.make_muscle_rig(nmuscle=muscles, seed=1003)
    layer = _gpu_layer(rig)
    limit = {29: 512, 63: 1024, 94: 1536, 131: 2048}
    assert all(layer._torque_entries.nentry <= limit[m] if m in limit else layer._torque_entries.nentry > limit[m - 1] for m in [muscles])
    entries = (layer._torque_entries, layer._muscle_entries, layer._moment_entries)
    stated = [e.nother for e in entries]
    for nworld in (70, 1537, 3601):
        ctx_d = torch.from_numpy(synth.make_muscle_context(rig, nworld, seed=6)).cuda()
        act = torch.rand(nworld, rig.muscle_count, device="cuda")
        act[:, ::7] = 0.0
        g = torch.randn(nworld, rig.torque_dim, device="cuda")

        def run():
            mean, _, unit = layer._warp_muscle_dynamics_from_activation_forward(act, ctx_d, include_passive_force=True)
            lo, hi = layer._compute_activation_torque_bounds_warp(ctx_d, select_active=False)
            return mean, layer._warp_muscle_dynamics_from_activation_backward(ctx_d, g), layer.eval_muscle_sparse_moment(ctx_d), lo, hi

        got = run()
        for e in entries:
            e.nother = 0
        for a, b in zip(got, run()):
            assert torch.equal(a, b)
        for e, n in zip(entries, stated):
            e.nother = n


def test_packed_entries_are_the_list_in_another_order():
    """Kinds together, the first two in whole wavefronts, every entry once; lists with other coefficients are refused."""
    layer = MuscleDynamicsLayer((rig := synth.make_muscle_rig(nmuscle=50, seed=3)).topology, **rig.dims(), device="cpu")
    _, torque, segment, muscle, a, b = layer.torque_entries_host
    words, counts = pack_context_entries(segment, torque, muscle, a, b)
    assert counts[0] % 64 == 0 and counts[1] % 64 == 0 and sum(counts) == len(words)
    place = words[:, 1] & 0xFFFF
    real = place < len(segment)
    assert np.array_equal(np.sort(place[real]), np.arange(len(segment))) and (place[~real] == len(segment)).all()
    at = place[real]
    assert np.array_equal(words[real, 0], (segment[at] | torque[at] << 16).astype(np.uint32)) and np.array_equal(words[real, 1] >> 16, muscle[at])
    kind = np.repeat([0, 1, 2], counts)[real]
    assert np.array_equal(a[at], np.float32([0, 1, 1])[kind]) and np.array_equal(b[at], np.float32([1, 0, 1])[kind])
    assert pack_context_entries(segment, torque, muscle, a * 0.5, b) is None


@pytest.mark.gpu
@pytest.mark.parametrize("muscles", [3, 74, 76, 158, 164, 225, 226, 320, 325])
@pytest.mark.parametrize("swap", [False, True, "some"])
def test_gpu_from_context_equals_waypoints_and_forces_in_memory(muscles, swap):
    """Torque, gradient and moment in one launch: the bits of the kernels with waypoints and forces in
    memory, on both sides of 1280, 2560, 3584 and 5120 entries (128, 256 and 512 threads; more than a workgroup keeps), for segments that
    run up the tree, down it and, in one list, both, one world and several per workgroup, and with poses, centres and axes that are not finite."""
    rig = synth.make_muscle_rig(nmuscle=muscles, seed=1003)
    t = rig.topology
    if swap:  # the end's body above the start's: entries with a start coefficient alone
        on = np.arange(len(t.apply_segment_start_idx)) % 3 != 0 if swap == "some" else True
        pick = lambda a, b: np.where(on, np.asarray(b), np.asarray(a))  # noqa: E731
        t = dataclasses.replace(
            t, apply_segment_start_idx=pick(t.apply_segment_start_idx, t.apply_segment_end_idx),
            apply_segment_end_idx=pick(t.apply_segment_end_idx, t.apply_segment_start_idx),
            apply_segment_body_start_idx=pick(t.apply_segment_body_start_idx, t.apply_segment_body_end_idx),
            apply_segment_body_end_idx=pick(t.apply_segment_body_end_idx, t.apply_segment_body_start_idx),
        )  # fmt: skip
    layer = MuscleDynamicsLayer(t, **rig.dims(), mechanics=MuscleMechanics(), device="cuda")
    kinds = [c.kind_count[:2] for c in layer._context if c is not None]
    assert all((k[0] > 0) == (swap is not True) and (k[1] > 0) == bool(swap) for k in kinds)
    assert (layer._context[0] is None) == (muscles == 325) and (layer._context[1] is None) == (layer._context[2] is None) == (muscles == 325)
    entries = (layer._torque_entries, layer._muscle_entries, layer._moment_entries)
    stated = [e.nother for e in entries]
    for nworld, odd in ((1, False), (1901, False), (67, True)):
        ctx = synth.make_muscle_context(rig, nworld, seed=6)
        if odd:
            for k, v in enumerate((np.inf, -np.inf, np.nan, 3.0e38)):
                ctx[8 * k + 1, layer._com_off + 3 + k % 3] = v
                ctx[8 * k + 2, layer._cdof_off + 6 * (layer.root_dof_count + k) + k] = v
                ctx[8 * k + 3, 3 * (k + 1)] = v
        ctx_d = torch.from_numpy(np.pad(ctx, ((0, 0), (0, 5)))).cuda()[:, : ctx.shape[1] + 2]
        act = torch.rand(nworld, rig.muscle_count, device="cuda")
        act[:, ::7] = 0.0
        g = torch.randn(nworld, rig.torque_dim, device="cuda")

        def run():
            return [layer._torque_from_context(act, ctx_d, passive) for passive in (False, True)] + [
                layer._warp_muscle_dynamics_from_activation_backward(ctx_d, g), layer.eval_muscle_sparse_moment(ctx_d)]  # fmt: skip

        got = run()
        for e in entries:
            e.nother = 0
        for a, b in zip(got, run()):
            assert torch.equal(torch.nan_to_num(a, 1.0, 2.0, 3.0), torch.nan_to_num(b, 1.0, 2.0, 3.0)) and torch.equal(a.isnan(), b.isnan())
        for e, n in zip(entries, stated):
            e.nother = n


@pytest.mark.parametrize("muscles", [1, 8, 50])
@pytest.mark.parametrize("swap", [False, True])
def test_groups_are_the_list_in_another_order(muscles, swap):
    """Every entry once, three to a group at most, alike in segment and kind (the moment: in row, in the row's order),
    64 groups of a kind and number together, fills in the list's place behind its last."""
    layer = MuscleDynamicsLayer((rig := synth.make_muscle_rig(nmuscle=muscles, seed=3)).topology, **rig.dims(), device="cpu")
    _, torque, segment, muscle, a, b = layer.torque_entries_host
    if swap:
        a, b = np.where(segment % 2, a, b), np.where(segment % 2, b, a)
    kind, n = np.where(a == 0, 0, np.where(b == 0, 1, 2)), len(segment)
    words, kinds = group_context_entries(segment, torque, muscle, a, b)
    assert len(words) == 64 * len(kinds)
    of = np.repeat(kinds, 64)
    place = np.stack([words[:, 2] >> 16, words[:, 3] & 0xFFFF, words[:, 3] >> 16], 1)
    dof = np.stack([words[:, 0] >> 16, words[:, 1] & 0xFFFF, words[:, 1] >> 16], 1)
    used = place < n
    assert np.array_equal(np.sort(place[used]), np.arange(n)) and (place[~used] == n).all()
    assert all(used[g].sum() in (0, of[g] >> 2) and (used[g] == (np.arange(3) < used[g].sum())).all() for g in range(len(words)))
    group, slot = np.nonzero(used)
    at = place[group, slot]
    assert np.array_equal(words[group, 0] & 0xFFFF, segment[at]) and np.array_equal(dof[group, slot], torque[at])
    assert np.array_equal(words[group, 2] & 0xFFFF, muscle[at]) and np.array_equal(of[group] & 3, kind[at])

    e = layer.sparse_entries
    off, seg = e.muscle_dof_segment_offsets, np.asarray(e.segment_idx)
    words, kinds = group_context_rows(off, seg, e.muscle_dof_torque_idx, e.start_coeff, e.end_coeff)
    row, of = words[:, 0] >> 16, np.repeat(kinds, 64)
    real = row < len(off) - 1
    assert np.array_equal(np.sort(row[real]), np.arange(len(off) - 1)) and (row[~real] == len(seg)).all()
    for g in np.flatnonzero(real):
        k = np.arange(off[row[g]], off[row[g] + 1])
        assert words[g, 0] & 0xFFFF == e.muscle_dof_torque_idx[row[g]]
        assert [words[g, 1] & 0xFFFF, words[g, 1] >> 16, words[g, 2]][: len(k)] == seg[k].tolist()
        want = [0 if e.start_coeff[i] == 0 else 1 if e.end_coeff[i] == 0 else 2 for i in k] + [3] * (3 - len(k))
        assert of[g] == want[0] | want[1] << 2 | want[2] << 4
    longer = np.concatenate([off[:-1], [off[-1] + 4]])
    assert group_context_rows(longer, np.append(seg, [0] * 4), e.muscle_dof_torque_idx, np.append(e.start_coeff, [1.0] * 4), np.append(e.end_coeff, [1.0] * 4)) is None


@pytest.mark.parametrize("what", [0, 1, 2])
def test_a_world_that_fills_64_kb_goes_from_its_context(what):
    """The words of a world, entries with four behind them, segments, axes, forces, centres and two flags, up to the limit
    and one past it (nworld = 0 only checks the sizes)."""
    import ctypes as C

    from instantmimic_amd import _lib

    sizes = dict(nbody=23, nwaypoint=900, nsegment=1160, ntorque=61, nmuscle=500)
    rest = 9 * sizes["nsegment"] + 7 * sizes["ntorque"] + sizes["nmuscle"] + 3 * sizes["nbody"] + 2
    for over in (0, 1):
        n = 16384 + over - rest - 4
        c = _lib.MuscleContext(ld_params=4, nrow=60, nentry=n, npacked=n, kind_count=(C.c_int32 * 3)(0, 0, n), **sizes)
        assert n <= 5120
        status = _lib.lib().im_muscle_from_context(C.byref(c), what, None, 0, 6, None, 60, 0, None)
        assert status == (_lib.IM_ERR_UNSUPPORTED if over else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("muscles", [1, 57, 58, 64, 148, 149, 310, 314])
def test_gpu_groups_equal_the_list_entry_by_entry(muscles):
    """Groups and no groups on one context, on both sides of 512, 1024 and 2048 groups, where torque and gradient take
    the next number of threads or go entry by entry: the same bits, one world and several per workgroup."""
    rig = synth.make_muscle_rig(nmuscle=muscles, seed=1003)
    layer = _gpu_layer(rig)
    stated = [c.ngroup for c in layer._context]
    assert all(stated)
    for nworld in (1, 1701):
        ctx = torch.from_numpy(synth.make_muscle_context(rig, nworld, seed=8)).cuda()
        act = torch.rand(nworld, muscles, device="cuda")
        act[:, ::5] = 0.0
        g = torch.randn(nworld, rig.torque_dim, device="cuda")
        run = lambda: [layer._torque_from_context(act, ctx, p) for p in (False, True)] + [  # noqa: E731
            layer._warp_muscle_dynamics_from_activation_backward(ctx, g), layer.eval_muscle_sparse_moment(ctx)]  # fmt: skip
        got = run()
        for c in layer._context:
            c.ngroup = 0
        want = run()
        for c, n in zip(layer._context, stated):
            c.ngroup = n
        for x, y in zip(got, want):
            assert torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("muscles", [30, 40, 57, 58, 60, 65, 80, 90, 91, 128, 230, 231])
def test_gpu_groups_of_large_batches_equal_the_list_entry_by_entry(muscles):
    """Batches of a workgroup more than six, and than seven, for every compute unit: the rules between entries and groups, and
    five and six groups a thread up to their last size and beyond it; the same bits."""
    rig = synth.make_muscle_rig(nmuscle=muscles, seed=1003)
    layer = _gpu_layer(rig)
    stated = [c.ngroup for c in layer._context]
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    for nworld in (6 * ncu, 6 * ncu + 1, 7 * ncu + 1):
        ctx = torch.from_numpy(synth.make_muscle_context(rig, 67, seed=8)).cuda()[torch.arange(nworld, device="cuda") % 67].contiguous()
        act, g = torch.rand(nworld, muscles, device="cuda"), torch.randn(nworld, rig.torque_dim, device="cuda")
        run = lambda: [layer._torque_from_context(act, ctx, True), layer._warp_muscle_dynamics_from_activation_backward(ctx, g),  # noqa: E731
                       layer.eval_muscle_sparse_moment(ctx)]  # fmt: skip
        got = run()
        for c in layer._context:
            c.ngroup = 0
        want = run()
        for c, n in zip(layer._context, stated):
            c.ngroup = n
        for x, y in zip(got, want):
            assert torch.equal(x, y)


@pytest.mark.gpu
def test_gpu_torque_call_is_the_dispatchers_operator():
    """``ops.muscle_torque_forward`` in eager code with a gradient to record against the operator of that name through
    the dispatcher: values, gradients, what autograd refuses, what modes and hooks see."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from torch.utils.checkpoint import checkpoint

    rig = synth.make_muscle_rig(nmuscle=12, seed=3)
    layer = _gpu_layer(rig)
    key, nworld = ops.warp_op_key(layer), 33
    ctx = torch.from_numpy(synth.make_muscle_context(rig, nworld, seed=4)).cuda()
    act = torch.rand(nworld, 12, device="cuda", requires_grad=True)
    g = torch.randn(nworld, rig.torque_dim, device="cuda")
    many = torch.rand(2, nworld, 12, device="cuda")
    direct, dispatched = ops.muscle_torque_forward, torch.ops.instantmimic_muscle.torque_forward
    assert type(direct(act, ctx, key, True).grad_fn).__name__ != type(dispatched(act, ctx, key, True).grad_fn).__name__

    def outcome(f):
        try:
            return [t.detach().clone() for t in f()]
        except Exception as e:  # noqa: BLE001
            return type(e)

    def same(f):
        a, b = outcome(lambda: f(direct)), outcome(lambda: f(dispatched))
        if isinstance(a, type) or isinstance(b, type):
            assert a is b
        else:
            assert len(a) == len(b) and all(torch.equal(x, y) for x, y in zip(a, b))
        return a

    def twice(op):
        y = op(act, ctx, key, False)
        return [y, *torch.autograd.grad(y, act, g, retain_graph=True), *torch.autograd.grad(y, act, 2 * g)]

    def second(op):
        (ga,) = torch.autograd.grad(op(act, ctx, key, False), act, g.clone().requires_grad_(True), create_graph=True)
        return torch.autograd.grad(ga.sum(), act)

    def changed(op):
        c = ctx.clone()
        y = op(act, c, key, False)
        c.add_(1.0)
        return torch.autograd.grad(y, act, g)

    def context_gradient(op):
        c = ctx.clone().requires_grad_(True)
        return torch.autograd.grad(op(act, c, key, False).sum(), [act, c], allow_unused=True)[:1]

    assert not isinstance(same(twice), type)
    for f in (second, changed):
        assert issubclass(same(f), RuntimeError)
    same(context_gradient)
    same(lambda op: torch.autograd.grad(op(act, ctx, key, False), act, g, create_graph=True))
    same(lambda op: [torch.func.grad(lambda a: (op(a, ctx, key, False) * g).sum())(act.detach())])
    same(lambda op: [torch.func.vmap(lambda a: op(a, ctx, key, False))(many)])
    same(lambda op: [torch.autograd.grad(op(act, ctx, key, False), act, torch.stack([g, g]), is_grads_batched=True)[0]])
    same(lambda op: [torch.func.jvp(lambda a: op(a, ctx, key, False), (act.detach(),), (act.detach(),))[1]])
    same(lambda op: torch.autograd.grad(checkpoint(lambda a: op(a, ctx, key, True), act, use_reentrant=False), act, g))
    same(lambda op: [op(act.detach(), ctx, key, False), op(act.double(), ctx, key, False)])
    same(lambda op: [op(act[:, :5], ctx, key, False)])
    same(lambda op: [op(act, ctx[:, :9], key, False)])
    same(lambda op: [op(act, ctx, 10**9, False)])

    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Mode():
        direct(act, ctx, key, False)
    assert "instantmimic_muscle.torque_forward.default" in seen
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        y = direct(act, ctx, key, False)
    assert packed == [ctx.shape] and torch.equal(torch.autograd.grad(y, act, g)[0], same(twice)[1])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = direct(act, ctx, key, False)
        got = torch.autograd.grad(y, act, g)[0]
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, same(twice)[1])


def _in_a_process_of_its_own(script: str) -> None:
    """What is registered with an operator, or taken from torch, stays so for the process."""
    import subprocess
    import sys

    from conftest import ROOT

    done = subprocess.run([sys.executable, "-c", script], cwd=ROOT, capture_output=True, text=True, timeout=110)
    assert done.returncode == 0, done.stdout + done.stderr


@pytest.mark.parametrize("take", ["del torch._C._dispatch_keys", "del torch._C._functorch.peek_interpreter_stack", "del torch.autograd.forward_ad._current_level",
                                  "torch._C._dispatch_has_kernel_for_any_dispatch_key = lambda name: False"])  # fmt: skip
def test_torque_operator_without_a_private_name_of_torch(take):
    _in_a_process_of_its_own(f"""
import torch
{take}
from instantmimic_amd.muscle import warp_custom_ops as ops
assert ops._EAGER is None
assert type(ops.muscle_torque_forward) is type(ops.muscle_torque_backward) is torch.library.CustomOpDef
""")


def test_torque_operator_notices_what_is_registered_with_it():
    _in_a_process_of_its_own("""
import torch
from instantmimic_amd.muscle import warp_custom_ops as ops
forward, backward = ops.muscle_torque_forward, ops.muscle_torque_backward
assert ops._is_as_defined(forward) and ops._is_as_defined(backward)
for key in ("CUDA", "AutocastCUDA", "AutogradCUDA"):
    lib = torch.library.Library(ops.NAMESPACE, "IMPL")
    lib.impl("torque_forward", lambda *a: None, key)
    assert not ops._is_as_defined(forward) and ops._is_as_defined(backward)
    lib._destroy()
    assert ops._is_as_defined(forward)
torch.library.register_autocast("instantmimic_muscle::torque_backward", "cuda", torch.float16)
assert not ops._is_as_defined(backward) and ops._is_as_defined(forward)
forward.register_autocast("cuda", torch.float16)
assert not ops._is_as_defined(forward)
""")
    for register in ('register_kernel("cuda", lambda *a: None)', 'register_kernel(None, lambda *a: None)', "register_autograd(lambda ctx, g: g)"):
        _in_a_process_of_its_own(f"""
from instantmimic_amd.muscle import warp_custom_ops as ops
ops.muscle_torque_forward.{register}
assert not ops._is_as_defined(ops.muscle_torque_forward)
""")


@pytest.mark.gpu
def test_gpu_torque_call_under_a_registered_cast():
    """With a gradient to record as without, and in the backward."""
    _in_a_process_of_its_own("""
import torch
from instantmimic_amd import synth
from instantmimic_amd.muscle import warp_custom_ops as ops
from instantmimic_amd.muscle.muscle_dynamics import MuscleDynamicsLayer
rig = synth.make_muscle_rig(nmuscle=12, seed=3)
layer = MuscleDynamicsLayer(rig.topology, **rig.dims(), device="cuda")
key, ctx = ops.warp_op_key(layer), torch.from_numpy(synth.make_muscle_context(rig, 33, seed=4)).cuda()
act, g = torch.rand(33, 12, device="cuda", requires_grad=True), torch.randn(33, rig.torque_dim, device="cuda")
direct, dispatched = ops.muscle_torque_forward, torch.ops.instantmimic_muscle.torque_forward
def both(op):
    with torch.autocast("cuda", torch.float16):
        y = op(act, ctx, key, False)
        return y.detach(), torch.autograd.grad(y, act, g)[0]
def same(a, b):
    return all(x.dtype == y.dtype and torch.equal(x, y) for x, y in zip(a, b))
plain = both(direct)
assert same(plain, both(dispatched))
ops.muscle_torque_backward.register_autocast("cuda", torch.float16)
assert same(both(direct), both(dispatched))
direct.register_autocast("cuda", torch.float16)
cast = both(direct)
assert same(cast, both(dispatched)) and not torch.equal(cast[0], plain[0])
""")
