"""Muscle moment-arm contractions: host tables, oracle pinning (CPU) and GPU parity."""

import numpy as np
import pytest

from instantmimic_amd import synth
from instantmimic_amd.muscle import muscle_qfrc_projector as Q
from oracle import ref as R


def _setup(nworld):
    mb = synth.make_muscles(nworld)
    rowadr, rownnz, colind = synth.csr_from_parents(synth.snu_parents())
    ent = Q.entries_from_muscle_dofs(mb.muscle_dofs, mb.nmuscle)
    np.testing.assert_array_equal(np.stack([ent.muscle_dof_muscle_idx, ent.muscle_dof_torque_idx], 1), mb.muscle_dofs)
    nv = len(rowadr)
    offsets, order = Q.torque_sorted_entries(ent.muscle_dof_torque_idx, nv - mb.root_dof_count)
    prepared = Q.prepare_muscle_implicit_qderiv_pairs(
        pair_entry_i=ent.pair_entry_i, pair_entry_j=ent.pair_entry_j, pair_muscle_idx=ent.pair_muscle_idx,
        muscle_dof_torque_idx=ent.muscle_dof_torque_idx, matrix_elemid=synth.matrix_elemid(rowadr, rownnz, colind),
        root_dof_count=mb.root_dof_count,
    )  # fmt: skip
    return mb, (rowadr, rownnz, colind), ent, offsets, order, prepared


def test_tables_by_brute_force():
    mb, st, ent, offsets, order, prepared = _setup(1)
    # entries sorted by (muscle, dof); every muscle's pairs are its lower triangle
    key = ent.muscle_dof_muscle_idx.astype(np.int64) * 1000 + ent.muscle_dof_torque_idx
    assert (np.diff(key) > 0).all()
    expect = [(i, j, m) for m in range(mb.nmuscle) for i in range(ent.muscle_dof_offsets[m], ent.muscle_dof_offsets[m + 1]) for j in range(ent.muscle_dof_offsets[m], i + 1)]
    got = list(zip(ent.pair_entry_i.tolist(), ent.pair_entry_j.tolist(), ent.pair_muscle_idx.tolist()))
    assert got == expect
    # torque-sorted order: ascending entry index within a dof
    for j in range(len(offsets) - 1):
        e = order[offsets[j] : offsets[j + 1]]
        assert (ent.muscle_dof_torque_idx[e] == j).all() and (np.diff(e) > 0).all()
    # muscles stay on one chain, so nothing is dropped
    assert prepared.dropped_pair_count == 0
    tables = Q.gather_tables(prepared, ent.muscle_dof_muscle_idx)
    elem_ids, chunk_offsets, chunk_pairs, nentry, chunk_count = tables
    packed = chunk_pairs.reshape(16, chunk_count)
    seen = []
    for slot, elem in enumerate(elem_ids):
        for c in range(chunk_offsets[slot], chunk_offsets[slot + 1]):
            for k in range(16):
                i, j = packed[k, c] & 0xFFFF, packed[k, c] >> 16
                if i < nentry:
                    seen.append((int(elem), int(i), int(j)))
    want = sorted(zip(prepared.pair_elem_id.tolist(), prepared.pair_entry_i.tolist(), prepared.pair_entry_j.tolist()))
    assert sorted(seen) == want and len(seen) == len(want)
    # pairs off M's pattern are dropped: couple two branches artificially
    bad = Q.prepare_muscle_implicit_qderiv_pairs(
        pair_entry_i=[1], pair_entry_j=[0], pair_muscle_idx=[0], muscle_dof_torque_idx=[0, 10],
        matrix_elemid=synth.matrix_elemid(*st), root_dof_count=6,
    )  # fmt: skip
    assert bad.dropped_pair_count == 1 and bad.pair_elem_id.size == 0


def _dense_a(mb, nv):
    A = np.zeros((mb.moment.shape[0], mb.nmuscle, nv))
    A[:, mb.muscle_dofs[:, 0], mb.muscle_dofs[:, 1] + mb.root_dof_count] = mb.moment
    return A


def test_oracle_against_dense_fp64():
    mb, st, ent, offsets, order, prepared = _setup(24)
    nv = len(st[0])
    A = _dense_a(mb, nv)
    tau = R.muscle_project(mb.moment, mb.force, offsets, order, ent.muscle_dof_muscle_idx, mb.root_dof_count, nv)
    tau64 = np.einsum("wmj,wm->wj", A, mb.force.astype(np.float64))
    assert R.rel_l2(tau, tau64) < 1e-6
    assert np.abs(tau[:, : mb.root_dof_count]).max() == 0.0
    elem_ids, chunk_offsets, chunk_pairs, nentry, chunk_count = Q.gather_tables(prepared, ent.muscle_dof_muscle_idx)
    q0 = np.random.default_rng(3).normal(size=(24, len(st[2]))).astype(np.float32)
    q = R.muscle_implicit_gather(mb.moment, mb.slope, ent.muscle_dof_muscle_idx, elem_ids, chunk_offsets, chunk_pairs, chunk_count, mb.timestep, q0)
    dense = np.einsum("wmi,wm,wmj->wij", A, mb.slope.astype(np.float64), A) * mb.timestep
    rowi = R.rows_of(st[1])
    want = q0 + dense[:, rowi, np.asarray(st[2])]
    assert R.rel_l2(q, want) < 1e-6
    # linear in the slope: doubling it doubles the added term exactly (power of two)
    zero = np.zeros_like(q0)
    q1 = R.muscle_implicit_gather(mb.moment, mb.slope, ent.muscle_dof_muscle_idx, elem_ids, chunk_offsets, chunk_pairs, chunk_count, mb.timestep, zero)
    q2 = R.muscle_implicit_gather(mb.moment, 2 * mb.slope, ent.muscle_dof_muscle_idx, elem_ids, chunk_offsets, chunk_pairs, chunk_count, mb.timestep, zero)
    np.testing.assert_array_equal(q2, 2 * q1)


@pytest.mark.gpu
@pytest.mark.parametrize("nworld", [1, 130, 4096])
def test_gpu_matches_oracle_bitwise(device, nworld):
    import torch

    mb, st, ent, offsets, order, prepared = _setup(nworld)
    nv = len(st[0])
    t = lambda a, dt=None: torch.from_numpy(np.ascontiguousarray(a if dt is None else a.astype(dt))).to(device)  # noqa: E731
    moment, force, slope = t(mb.moment), t(mb.force), t(mb.slope)
    qfrc = torch.full((nworld, nv + 3), 7.0, device=device)
    Q.project_muscle_sparse_moment_qfrc(moment, force, t(offsets, np.int32), t(order, np.int32), t(ent.muscle_dof_muscle_idx, np.int32), mb.root_dof_count, qfrc[:, :nv])
    gather = Q.build_muscle_implicit_qderiv_gather(prepared, ent.muscle_dof_muscle_idx, device)
    assert gather is not None
    q0 = np.random.default_rng(3).normal(size=(nworld, len(st[2]))).astype(np.float32)
    qd = t(q0)
    Q.apply_muscle_implicit_qderiv_gather(gather, moment, slope, mb.timestep, qd)
    torch.cuda.synchronize()
    tau_ref = R.muscle_project(mb.moment, mb.force, offsets, order, ent.muscle_dof_muscle_idx, mb.root_dof_count, nv)
    got = qfrc.cpu().numpy()
    np.testing.assert_array_equal(got[:, mb.root_dof_count : nv], tau_ref[:, mb.root_dof_count :])
    assert (got[:, : mb.root_dof_count] == 7.0).all() and (got[:, nv:] == 7.0).all()  # root dofs and padding untouched
    tables = Q.gather_tables(prepared, ent.muscle_dof_muscle_idx)
    q_ref = R.muscle_implicit_gather(mb.moment, mb.slope, ent.muscle_dof_muscle_idx, tables[0], tables[1], tables[2], tables[4], mb.timestep, q0)
    np.testing.assert_array_equal(qd.cpu().numpy(), q_ref)
    # the contract's bound as well
    assert R.rel_l2(got[:, mb.root_dof_count : nv], tau_ref[:, mb.root_dof_count :]) <= 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("nworld", [511, 512, 513, 2047, 2048, 2049])
@pytest.mark.parametrize("nmuscle", [20, 40, 420, 1100])
def test_gpu_gather_of_two_worlds_a_workgroup(device, nmuscle, nworld):
    """Both sides of the batch from which a workgroup takes two worlds (two for every compute unit), with a world left over,
    on 256 threads (20 muscles) and on 512, and where a unit does not hold two such workgroups (1100): the oracle's bits, and
    the columns beside the matrix stay as they are."""
    import torch

    mb = synth.make_muscles(nworld, nmuscle=nmuscle, seed=5)
    rowadr, rownnz, colind = synth.csr_from_parents(synth.snu_parents())
    ent = Q.entries_from_muscle_dofs(mb.muscle_dofs, mb.nmuscle)
    prepared = Q.prepare_muscle_implicit_qderiv_pairs(
        pair_entry_i=ent.pair_entry_i, pair_entry_j=ent.pair_entry_j, pair_muscle_idx=ent.pair_muscle_idx,
        muscle_dof_torque_idx=ent.muscle_dof_torque_idx, matrix_elemid=synth.matrix_elemid(rowadr, rownnz, colind),
        root_dof_count=mb.root_dof_count,
    )  # fmt: skip
    gather = Q.build_muscle_implicit_qderiv_gather(prepared, ent.muscle_dof_muscle_idx, device)
    q0 = np.random.default_rng(3).normal(size=(nworld, len(colind))).astype(np.float32)
    wide = torch.full((nworld, len(colind) + 3), 7.0, device=device)
    wide[:, :-3] = torch.from_numpy(q0).to(device)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    Q.apply_muscle_implicit_qderiv_gather(gather, t(mb.moment), t(mb.slope), mb.timestep, wide[:, :-3])
    tables = Q.gather_tables(prepared, ent.muscle_dof_muscle_idx)
    want = R.muscle_implicit_gather(mb.moment, mb.slope, ent.muscle_dof_muscle_idx, tables[0], tables[1], tables[2], tables[4], mb.timestep, q0)
    np.testing.assert_array_equal(wide[:, :-3].cpu().numpy(), want)
    assert (wide[:, -3:] == 7.0).all()


@pytest.mark.gpu
def test_gpu_projection_with_more_entries_than_one_staging_trip(device):
    """420 muscles give about 1900 entries: several of a thread's twelve places stay empty in the
    projection kernel's trip through LDS (the sizes beyond one trip are tested below)."""
    import torch

    nworld = 97
    mb = synth.make_muscles(nworld, nmuscle=420, seed=5)
    rowadr, _, _ = synth.csr_from_parents(synth.snu_parents())
    nv = len(rowadr)
    ent = Q.entries_from_muscle_dofs(mb.muscle_dofs, mb.nmuscle)
    assert len(ent.muscle_dof_torque_idx) > 1536
    offsets, order = Q.torque_sorted_entries(ent.muscle_dof_torque_idx, nv - mb.root_dof_count)
    t = lambda a, dt=None: torch.from_numpy(np.ascontiguousarray(a if dt is None else a.astype(dt))).to(device)  # noqa: E731
    qfrc = torch.full((nworld, nv), 7.0, device=device)
    Q.project_muscle_sparse_moment_qfrc(t(mb.moment), t(mb.force), t(offsets, np.int32), t(order, np.int32), t(ent.muscle_dof_muscle_idx, np.int32), mb.root_dof_count, qfrc)
    torch.cuda.synchronize()
    tau_ref = R.muscle_project(mb.moment, mb.force, offsets, order, ent.muscle_dof_muscle_idx, mb.root_dof_count, nv)
    got = qfrc.cpu().numpy()
    np.testing.assert_array_equal(got[:, mb.root_dof_count :], tau_ref[:, mb.root_dof_count :])
    assert (got[:, : mb.root_dof_count] == 7.0).all()


def _fv_case(nworld, seed=4, active_type=1.0, nmuscle=37, points=(2, 6), dofs=(1, 4)):
    """Random muscles over random waypoints: every branch of the force-velocity curve is hit."""
    rng = np.random.default_rng(seed)
    nv, root = 30, 6
    counts = rng.integers(*points, nmuscle)
    wp_start = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    nwp = int(wp_start[-1])
    waypoints = rng.normal(size=(nworld, nwp, 3)).astype(np.float32)
    ndof = rng.integers(*dofs, nmuscle)
    dof_offsets = np.concatenate([[0], np.cumsum(ndof)]).astype(np.int32)
    dof_torque = np.concatenate([np.sort(rng.choice(nv - root, n, replace=False)) for n in ndof]).astype(np.int32)
    params = np.stack([rng.uniform(100, 3000, nmuscle), rng.uniform(0.5, 1.5, nmuscle), rng.uniform(0.0, 0.5, nmuscle), rng.uniform(0, 0.5, nmuscle)], 1).astype(np.float32)
    rest = rng.uniform(2.0, 6.0, nmuscle).astype(np.float32)
    scale = rng.uniform(0.1, 0.5, nmuscle).astype(np.float32)
    act = rng.uniform(-0.2, 1.3, (nworld, nmuscle)).astype(np.float32)
    qvel = rng.normal(scale=3.0, size=(nworld, nv)).astype(np.float32)
    moment = rng.normal(scale=0.2, size=(nworld, int(dof_offsets[-1]))).astype(np.float32)
    model = np.array([1.2, 0.4, 1.6, active_type, 0.5 if active_type else 0.45, 1.6, 0, 0, 0], np.float32)
    fv = np.array([1.5, 1.4, 1.0, 1.0], np.float32)
    return dict(waypoints=waypoints, wp_start=wp_start, params=params, rest=rest, length_scale=scale, act=act, qvel=qvel,
                moment=moment, dof_offsets=dof_offsets, dof_torque=dof_torque, root=root, model=model, fv=fv)  # fmt: skip


def _fv64(c):
    """The same state in fp64 NumPy, written from the formulas (muscle_qfrc_projector.py:2505-2570)."""
    wp = c["waypoints"].astype(np.float64)
    nworld, nmuscle = wp.shape[0], len(c["wp_start"]) - 1
    seg = np.linalg.norm(np.diff(wp, axis=1), axis=2)
    out = np.zeros((5, nworld, nmuscle))
    vmax, fvmax, clamp, inc = (float(v) for v in c["fv"])
    for m in range(nmuscle):
        a, b = c["wp_start"][m], c["wp_start"][m + 1]
        length = seg[:, a : b - 1].sum(1)
        e0, e1 = c["dof_offsets"][m], c["dof_offsets"][m + 1]
        vel = -(c["moment"][:, e0:e1].astype(np.float64) * c["qvel"][:, c["dof_torque"][e0:e1] + c["root"]]).sum(1)
        vs = max(float(c["length_scale"][m]) * vmax, 1e-6)
        v, y = vel / vs, fvmax - 1.0
        mult = np.where(v <= -1, 0.0, np.where(v <= 0, (v + 1) ** 2, np.where(v <= y, fvmax - (y - v) ** 2 / y, fvmax)))
        slope = np.where(v <= -1, 0.0, np.where(v <= 0, 2 * (v + 1), np.where(v <= y, 2 * (y - v) / y, 0.0)))
        act = np.clip(c["act"][:, m].astype(np.float64), 0, 1) if clamp else c["act"][:, m]
        f0, lm0, lt0, pen = (float(x) for x in c["params"][m])
        ln = np.clip((length / max(float(c["rest"][m]), 1e-6) - lt0) / max(lm0, 1e-6), float(c["model"][1]), float(c["model"][2]))
        lmin, lmax = float(c["model"][4]), float(c["model"][5])  # MuJoCo piecewise-quadratic active curve
        lo, hi = 0.5 * (lmin + 1), 0.5 * (1 + lmax)
        fl = np.where((ln < lmin) | (ln > lmax), 0.0, np.where(ln <= lo, 0.5 * ((ln - lmin) / (lo - lmin)) ** 2, np.where(
            ln <= 1, 1 - 0.5 * ((1 - ln) / (1 - lo)) ** 2, np.where(ln <= hi, 1 - 0.5 * ((ln - 1) / (hi - 1)) ** 2, 0.5 * ((lmax - ln) / (lmax - hi)) ** 2))))  # fmt: skip
        unit = f0 * fl * np.cos(pen) * float(c["model"][0])
        out[:, :, m] = length, act * mult, vel, mult, inc * act * unit * slope / vs
    return out


def test_force_velocity_state_oracle_against_fp64():
    c = _fv_case(50)
    got = np.stack(R.muscle_force_velocity_state(**c))
    want = _fv64(c)
    for k, name in enumerate(("length", "effective activation", "velocity", "multiplier", "slope")):
        np.testing.assert_allclose(got[k], want[k], rtol=3e-5, atol=3e-5 * max(1.0, np.abs(want[k]).max()), err_msg=name)
    v = want[2] / np.maximum(c["length_scale"] * 1.5, 1e-6)
    assert (v <= -1).any() and ((v > -1) & (v <= 0)).any() and ((v > 0) & (v <= 0.4)).any() and (v > 0.4).any()
    assert (c["act"] < 0).any() and (got[1] >= 0).all()  # clamped activation


@pytest.mark.gpu
@pytest.mark.parametrize("active_type", [1.0, 0.0])
def test_gpu_force_velocity_state(device, active_type):
    """im_muscle_force_velocity_state against the oracle: length, velocity, multiplier and effective
    activation bit for bit; the slope carries cosf (and expf with the gaussian active curve), which
    differ by a few ulp between libm and the GPU, and is held to 2e-6."""
    import torch

    c = _fv_case(130, active_type=active_type)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    outs = [torch.full((130, 37), float("nan"), device=device) for _ in range(5)]
    Q.eval_muscle_force_velocity_state(
        t(c["waypoints"]), t(c["wp_start"]), t(c["params"]), t(c["rest"]), t(c["length_scale"]), t(c["act"]), t(c["qvel"]),
        t(c["moment"]), t(c["dof_offsets"]), t(c["dof_torque"]), c["root"], muscle_force_scale=float(c["model"][0]),
        muscle_length_norm_min=float(c["model"][1]), muscle_length_norm_max=float(c["model"][2]), vmax=1.5, fvmax=1.4,
        clamp_activation=True, include_active=True, active_force_model_params=c["model"][3:6],
        muscle_length=outs[0], effective_activation=outs[1], length_velocity=outs[2], force_velocity_multiplier=outs[3],
        force_velocity_slope=outs[4],
    )  # fmt: skip
    torch.cuda.synchronize()
    want = R.muscle_force_velocity_state(**c)
    for k in range(4):
        np.testing.assert_array_equal(outs[k].cpu().numpy(), want[k])
    np.testing.assert_allclose(outs[4].cpu().numpy(), want[4], rtol=2e-6, atol=1e-6 * np.abs(want[4]).max())
    assert (want[4] == 0).any() and (want[4] != 0).any()
    np.testing.assert_array_equal(outs[4].cpu().numpy() == 0, want[4] == 0)  # the curve's flat parts are exact


@pytest.mark.gpu
@pytest.mark.parametrize("pad", [3, 12001])
def test_gpu_force_velocity_state_of_many_worlds(device, pad):
    """More worlds than resident workgroups, and rows that are columns of wider arrays (the last
    world's row ends with the array; the long stride asks for more than 64 KB of LDS): length, activation, velocity and multiplier bit for bit."""
    import torch

    n = 2100
    c = _fv_case(n, active_type=1.0)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731

    def wide(a):
        b = torch.full((a.shape[0], a.shape[1] + pad), float("nan"), device=device)
        b[:, pad:] = t(a)
        return b[:, pad:]

    outs = [torch.full((n, 37), float("nan"), device=device) for _ in range(5)]
    Q.eval_muscle_force_velocity_state(
        t(c["waypoints"]), t(c["wp_start"]), t(c["params"]), t(c["rest"]), t(c["length_scale"]), wide(c["act"]), t(c["qvel"]),
        wide(c["moment"]), t(c["dof_offsets"]), t(c["dof_torque"]), c["root"], muscle_force_scale=float(c["model"][0]),
        muscle_length_norm_min=float(c["model"][1]), muscle_length_norm_max=float(c["model"][2]), vmax=1.5, fvmax=1.4,
        clamp_activation=True, include_active=True, active_force_model_params=c["model"][3:6],
        muscle_length=outs[0], effective_activation=outs[1], length_velocity=outs[2], force_velocity_multiplier=outs[3],
        force_velocity_slope=outs[4],
    )  # fmt: skip
    want = R.muscle_force_velocity_state(**c)
    for k in range(4):
        np.testing.assert_array_equal(outs[k].cpu().numpy(), want[k])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1030, 3001])
@pytest.mark.parametrize("nmuscle", [1, 128, 129, 192, 193, 256, 257, 320, 321, 700])
def test_gpu_force_velocity_state_on_every_workgroup_size(device, nmuscle, n):
    """Both sides of the muscle counts at which a workgroup gets another 64 threads, more muscles than
    threads, workgroups that walk over several worlds: bit for bit."""
    import torch

    c = _fv_case(n, active_type=1.0, nmuscle=nmuscle)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    outs = [torch.full((n, nmuscle), float("nan"), device=device) for _ in range(5)]
    Q.eval_muscle_force_velocity_state(
        t(c["waypoints"]), t(c["wp_start"]), t(c["params"]), t(c["rest"]), t(c["length_scale"]), t(c["act"]), t(c["qvel"]),
        t(c["moment"]), t(c["dof_offsets"]), t(c["dof_torque"]), c["root"], muscle_force_scale=float(c["model"][0]),
        muscle_length_norm_min=float(c["model"][1]), muscle_length_norm_max=float(c["model"][2]), vmax=1.5, fvmax=1.4,
        clamp_activation=True, include_active=True, active_force_model_params=c["model"][3:6],
        muscle_length=outs[0], effective_activation=outs[1], length_velocity=outs[2], force_velocity_multiplier=outs[3],
        force_velocity_slope=outs[4],
    )  # fmt: skip
    want = R.muscle_force_velocity_state(**c)
    for k in range(4):
        np.testing.assert_array_equal(outs[k].cpu().numpy(), want[k])


@pytest.mark.gpu
@pytest.mark.parametrize("nmuscle, points, n", [(60, 18, 3), (60, 18, 1500), (200, 10, 1500), (350, 18, 1100)])
def test_gpu_force_velocity_state_of_short_and_long_muscles(device, nmuscle, points, n):
    """Muscles of no, one and up to sixteen distances and entries (both sums go four terms at a time with the next four
    asked for ahead), with the next world's rows held in registers and with muscles beyond the threads: bit for bit."""
    import torch

    c = _fv_case(n, seed=nmuscle, nmuscle=nmuscle, points=(1, points), dofs=(0, 17))
    assert {1, 2, 5, 6, 9} <= set(np.diff(c["wp_start"])) and {0, 1, 4, 5} <= set(np.diff(c["dof_offsets"]))
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    outs = [torch.full((n, nmuscle), float("nan"), device=device) for _ in range(5)]
    Q.eval_muscle_force_velocity_state(
        t(c["waypoints"]), t(c["wp_start"]), t(c["params"]), t(c["rest"]), t(c["length_scale"]), t(c["act"]), t(c["qvel"]),
        t(c["moment"]), t(c["dof_offsets"]), t(c["dof_torque"]), c["root"], muscle_force_scale=float(c["model"][0]),
        muscle_length_norm_min=float(c["model"][1]), muscle_length_norm_max=float(c["model"][2]), vmax=1.5, fvmax=1.4,
        clamp_activation=True, include_active=True, active_force_model_params=c["model"][3:6],
        muscle_length=outs[0], effective_activation=outs[1], length_velocity=outs[2], force_velocity_multiplier=outs[3],
        force_velocity_slope=outs[4],
    )  # fmt: skip
    want = R.muscle_force_velocity_state(**c)
    for k in range(4):
        np.testing.assert_array_equal(outs[k].cpu().numpy(), want[k])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 67])
@pytest.mark.parametrize("pad", [3, 12001])
def test_gpu_force_velocity_state_with_velocities_in_a_wider_array(device, n, pad):
    """The velocities as the last columns of a wider array, so that the last world's row ends with the
    allocation; poison in front of them: length, activation, velocity and multiplier bit for bit."""
    import torch

    c = _fv_case(n, active_type=1.0)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    wide = torch.full((n, c["qvel"].shape[1] + pad), float("nan"), device=device)
    wide[:, pad:] = t(c["qvel"])
    outs = [torch.full((n, 37), float("nan"), device=device) for _ in range(5)]
    Q.eval_muscle_force_velocity_state(
        t(c["waypoints"]), t(c["wp_start"]), t(c["params"]), t(c["rest"]), t(c["length_scale"]), t(c["act"]), wide[:, pad:],
        t(c["moment"]), t(c["dof_offsets"]), t(c["dof_torque"]), c["root"], muscle_force_scale=float(c["model"][0]),
        muscle_length_norm_min=float(c["model"][1]), muscle_length_norm_max=float(c["model"][2]), vmax=1.5, fvmax=1.4,
        clamp_activation=True, include_active=True, active_force_model_params=c["model"][3:6],
        muscle_length=outs[0], effective_activation=outs[1], length_velocity=outs[2], force_velocity_multiplier=outs[3],
        force_velocity_slope=outs[4],
    )  # fmt: skip
    want = R.muscle_force_velocity_state(**c)
    for k in range(4):
        np.testing.assert_array_equal(outs[k].cpu().numpy(), want[k])


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["column", "overlapping", "one row for all"])
def test_gpu_force_velocity_state_with_strides_shorter_than_a_row(device, layout):
    """Velocities and moments whose row stride is no row length: a transposed column (one world, stride
    1), windows into one array, one row for every world: bit for bit."""
    import torch

    n = 1 if layout == "column" else 5
    c = _fv_case(n, active_type=1.0)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731

    def laid_out(a):
        if layout == "column":
            return t(a[0]).as_strided(a.shape, (1, 1))
        step = 7 if layout == "overlapping" else 0
        flat = t(np.resize(a, a.shape[1] + step * n))
        return flat.as_strided((n, a.shape[1]), (step, 1))

    qvel, moment = laid_out(c["qvel"]), laid_out(c["moment"])
    assert qvel.stride(0) < qvel.shape[1]
    c["qvel"], c["moment"] = qvel.cpu().numpy().copy(), moment.cpu().numpy().copy()
    outs = [torch.full((n, 37), float("nan"), device=device) for _ in range(5)]
    Q.eval_muscle_force_velocity_state(
        t(c["waypoints"]), t(c["wp_start"]), t(c["params"]), t(c["rest"]), t(c["length_scale"]), t(c["act"]), qvel,
        moment, t(c["dof_offsets"]), t(c["dof_torque"]), c["root"], muscle_force_scale=float(c["model"][0]),
        muscle_length_norm_min=float(c["model"][1]), muscle_length_norm_max=float(c["model"][2]), vmax=1.5, fvmax=1.4,
        clamp_activation=True, include_active=True, active_force_model_params=c["model"][3:6],
        muscle_length=outs[0], effective_activation=outs[1], length_velocity=outs[2], force_velocity_multiplier=outs[3],
        force_velocity_slope=outs[4],
    )  # fmt: skip
    want = R.muscle_force_velocity_state(**c)
    for k in range(4):
        np.testing.assert_array_equal(outs[k].cpu().numpy(), want[k])


@pytest.mark.gpu
@pytest.mark.parametrize("muscles", [30, 690, 1950])
def test_gpu_projection_staging_sizes(device, muscles):
    """Rows shorter than eight terms, more than the 3072 entries of one staging trip, and more than
    64 KB of LDS: bit for bit."""
    import torch

    nworld = 33
    mb = synth.make_muscles(nworld, nmuscle=muscles, seed=5)
    nv = len(synth.csr_from_parents(synth.snu_parents())[0])
    ent = Q.entries_from_muscle_dofs(mb.muscle_dofs, mb.nmuscle)
    entries = len(ent.muscle_dof_torque_idx)
    assert muscles < 600 or entries > 3072
    assert muscles < 1900 or 4 * (2 * entries + muscles) > 65536 >= 4 * (entries + muscles) + 2 * (entries + 1)
    offsets, order = Q.torque_sorted_entries(ent.muscle_dof_torque_idx, nv - mb.root_dof_count)
    t = lambda a, dt=None: torch.from_numpy(np.ascontiguousarray(a if dt is None else a.astype(dt))).to(device)  # noqa: E731
    qfrc = torch.full((nworld, nv), 7.0, device=device)
    Q.project_muscle_sparse_moment_qfrc(t(mb.moment), t(mb.force), t(offsets, np.int32), t(order, np.int32), t(ent.muscle_dof_muscle_idx, np.int32), mb.root_dof_count, qfrc)
    want = R.muscle_project(mb.moment, mb.force, offsets, order, ent.muscle_dof_muscle_idx, mb.root_dof_count, nv)
    np.testing.assert_array_equal(qfrc.cpu().numpy()[:, mb.root_dof_count :], want[:, mb.root_dof_count :])


@pytest.mark.gpu
@pytest.mark.parametrize("entries", [511, 512, 513, 1024, 1025, 1536, 1537, 2048, 2049, 3072, 3073])
def test_gpu_projection_at_the_ends_of_a_trip(device, entries):
    """Both sides of the entry counts that a workgroup's one trip through LDS holds, with rows without an
    entry and one with most of them: bit for bit, root dofs and padding untouched."""
    import torch

    rng = np.random.default_rng(entries)
    nworld, nmuscle, ntorque, root = 5, 97, 21, 6
    dof = np.where(rng.uniform(size=entries) < 0.6, 3, rng.integers(0, ntorque, entries))
    dof[dof == 11] = 12
    offsets, order = Q.torque_sorted_entries(dof.astype(np.int32), ntorque)
    muscle = rng.integers(0, nmuscle, entries).astype(np.int32)
    moment, force = rng.normal(size=(nworld, entries)).astype(np.float32), rng.normal(size=(nworld, nmuscle)).astype(np.float32)
    t = lambda a, dt=None: torch.from_numpy(np.ascontiguousarray(a if dt is None else a.astype(dt))).to(device)  # noqa: E731
    qfrc = torch.full((nworld, root + ntorque + 2), 7.0, device=device)
    Q.project_muscle_sparse_moment_qfrc(t(moment), t(force), t(offsets, np.int32), t(order, np.int32), t(muscle), root, qfrc[:, : root + ntorque])
    want = R.muscle_project(moment, force, offsets, order, muscle, root, root + ntorque)
    got = qfrc.cpu().numpy()
    np.testing.assert_array_equal(got[:, root : root + ntorque], want[:, root:])
    assert (got[:, :root] == 7.0).all() and (got[:, root + ntorque :] == 7.0).all()
