"""Waypoint muscle layer on MI355X: pose context -> path geometry -> activation-to-torque
projection and its activation gradient.

Drop-in for the waypoint projection of the reference's ``MuscleDynamicsLayer``
(src/instantmimic/muscle/muscle_dynamics.py): static sparsity built as in
``muscle_qfrc_projector.py:336-510`` and ``muscle_dynamics.py:1318-1392``, raw context
layout of ``muscle_dynamics.py:4824-4838``, launch sequence of
``_warp_muscle_dynamics_from_activation_forward`` (:4958-5009 and the waypoint tail) and
``_warp_muscle_dynamics_from_activation_backward``.  Linear-blend-skinned attachments, the
force-velocity factor and the native body-wrench tiles of the reference are other paths of
that class and are not provided here; asking for them raises.

The arithmetic runs in ``libimhip``; tensors must live on the GPU.  Index tables are built
once on the host with NumPy.
"""

from __future__ import annotations

import ctypes as C
from dataclasses import dataclass

import numpy as np

from .. import _lib
from .muscle_qfrc_projector import MuscleDofSparseEntries, _np, build_muscle_dof_sparse_entries


@dataclass(frozen=True)
class MuscleMechanics:
    """The fields of the reference's MuscleMechanicsRuntimeSpec that the waypoint path reads
    (src/instantmimic/muscle/runtime_specs.py:66-96)."""

    force_scale: float = 1.0
    active_force_type: str = "gaussian"
    active_force_gamma: float = 0.45
    active_force_lmin: float = 0.5
    active_force_lmax: float = 1.6
    passive_force_type: str = "exponential"
    passive_force_k_pe: float = 5.5
    passive_force_e_mo: float = 0.3
    passive_force_lmax: float = 1.6
    passive_force_fpmax: float = 1.3
    length_norm_min: float = 0.2
    length_norm_max: float = 1.8
    include_passive_force_in_output: bool = False
    force_velocity_enabled: bool = False

    def __post_init__(self):
        # the reference's checks, muscle_dynamics.py:523-573
        if self.active_force_type not in {"gaussian", "mujoco"}:
            raise ValueError("muscle_active_force_type must be 'gaussian' or 'mujoco'")
        if self.active_force_gamma <= 0.0:
            raise ValueError("Gaussian active-force gamma must be positive")
        if not (0.0 < self.active_force_lmin < 1.0 and self.active_force_lmax > 1.0):
            raise ValueError("MuJoCo active-force lmin/lmax must satisfy 0 < lmin < 1 < lmax")
        if self.passive_force_type not in {"exponential", "mujoco"}:
            raise ValueError("muscle_passive_force_type must be 'exponential' or 'mujoco'")
        if self.passive_force_k_pe <= 0.0 or self.passive_force_e_mo <= 0.0:
            raise ValueError("exponential passive-force k_pe and e_mo must be positive")
        if self.passive_force_lmax <= 1.0 or self.passive_force_fpmax < 0.0:
            raise ValueError("MuJoCo passive-force lmax must exceed 1 and fpmax must be nonnegative")
        if self.force_velocity_enabled:
            raise NotImplementedError("the force-velocity factor is not part of this library")

    def active_params(self) -> tuple[float, float, float]:
        if self.active_force_type == "gaussian":
            return (0.0, self.active_force_gamma, 0.0)
        return (1.0, self.active_force_lmin, self.active_force_lmax)

    def passive_params(self) -> tuple[float, float, float]:
        if self.passive_force_type == "exponential":
            return (0.0, self.passive_force_k_pe, self.passive_force_e_mo)
        return (1.0, self.passive_force_lmax, self.passive_force_fpmax)


@dataclass(frozen=True)
class MuscleTopology:
    """The waypoint fields of the reference's MuscleTopologySpec (runtime_specs.py), as
    NumPy-convertible arrays."""

    muscle_params: np.ndarray  # (M, >= 4): f0, l_m0, l_t0, pennation
    muscle_rest_length: np.ndarray  # (M,)
    muscle_waypoints_local: np.ndarray  # (W, 3)
    muscle_waypoint_body: np.ndarray  # (W,)
    all_segment_muscle_idx: np.ndarray  # (S_all,) nondecreasing
    all_segment_start_idx: np.ndarray  # (S_all,) waypoint id; the end is start + 1
    apply_segment_muscle_idx: np.ndarray  # (S,)
    apply_segment_start_idx: np.ndarray
    apply_segment_end_idx: np.ndarray
    apply_segment_body_start_idx: np.ndarray
    apply_segment_body_end_idx: np.ndarray
    body_parentid: np.ndarray  # (nbody,)
    body_rootid: np.ndarray
    dof_bodyid: np.ndarray  # (>= full_torque_dim,)
    uses_lbs_waypoint_attachments: bool = False


def build_dof_subtree_mask(body_parentid, dof_bodyid, body_count: int, full_torque_dim: int) -> np.ndarray:
    """mask[dof, body] = 1 when the dof's body is the body or one of its ancestors below
    the world; world-body dofs move everything (muscle_qfrc_projector.py:336-356)."""
    parent = _np(body_parentid)
    ancestor = np.zeros((body_count, body_count), bool)
    for b in range(body_count):
        p = b
        while p != 0:
            ancestor[b, p] = True
            p = int(parent[p])
    dof_body = _np(dof_bodyid)[:full_torque_dim]
    mask = ancestor[:, dof_body].T.astype(np.float32)
    mask[dof_body == 0] = 1.0
    return mask


def build_muscle_segment_offsets(segment_muscle_idx, muscle_count: int) -> np.ndarray:
    """muscle_qfrc_projector.py:321-333"""
    counts = np.bincount(_np(segment_muscle_idx), minlength=muscle_count)
    return np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)


def build_torque_sparse_segment_entries(segment_start_dof_mask, segment_end_dof_mask, apply_segment_muscle_idx):
    """Per torque dof, the segments whose start or end coefficient is nonzero, ascending
    (muscle_qfrc_projector.py:378-456).  Returns offsets, torque, segment, muscle, start and
    end coefficient."""
    start = np.asarray(segment_start_dof_mask, np.float32)
    end = np.asarray(segment_end_dof_mask, np.float32)
    muscle = _np(apply_segment_muscle_idx)
    torque_idx, segment_idx = np.nonzero((start != 0) | (end != 0))  # row-major: torque, then segment
    offsets = np.concatenate([[0], np.cumsum(np.bincount(torque_idx, minlength=start.shape[0]))])
    return (
        offsets.astype(np.int32),
        torque_idx.astype(np.int32),
        segment_idx.astype(np.int32),
        muscle[segment_idx].astype(np.int32),
        start[torque_idx, segment_idx],
        end[torque_idx, segment_idx],
    )


def build_muscle_sparse_torque_entries(
    torque_entry_offsets, torque_segment_idx, torque_start_coeff, torque_end_coeff, apply_segment_muscle_idx,
    muscle_count: int,
):  # fmt: skip
    """The same entries sorted by (muscle, segment, torque) (muscle_qfrc_projector.py:459-510).
    Returns offsets, segment, torque, start and end coefficient."""
    offsets = _np(torque_entry_offsets)
    segment = _np(torque_segment_idx)
    if len(offsets) <= 1 or len(segment) == 0:
        z = np.zeros(0, np.int32)
        return np.zeros(muscle_count + 1, np.int32), z, z.copy(), np.zeros(0, np.float32), np.zeros(0, np.float32)
    torque = np.repeat(np.arange(len(offsets) - 1), np.diff(offsets))
    muscle = _np(apply_segment_muscle_idx)[segment]
    order = np.lexsort((torque, segment, muscle))
    return (
        build_muscle_segment_offsets(muscle, muscle_count),
        segment[order].astype(np.int32),
        torque[order].astype(np.int32),
        np.asarray(torque_start_coeff, np.float32)[order],
        np.asarray(torque_end_coeff, np.float32)[order],
    )


# What im_muscle_from_context computes
_TORQUE, _GRAD, _MOMENT = 0, 1, 2


def pack_context_entries(segment, torque, muscle, start_coeff, end_coeff):
    """A list of (segment, dof) entries in the packed order of im_muscle_from_context: the entries of a
    kind (end only, start only, both) together, the first two kinds filled up to whole wavefronts.
    Returns (packed (n, 2) uint32, counts of the kinds), or None where a coefficient is neither 0 nor 1 or
    a number does not fit 16 bits."""
    segment, torque, muscle = (np.asarray(a, np.int64) for a in (segment, torque, muscle))
    a, b, n = np.asarray(start_coeff), np.asarray(end_coeff), len(segment)
    if n == 0 or n >= 65535 or max(segment.max(), torque.max(), muscle.max()) >= 65536:
        return None
    if not (((a == 0) | (a == 1)) & ((b == 0) | (b == 1)) & (a + b > 0)).all():
        return None
    words, counts = [], []
    for kind, on in enumerate(((a == 0) & (b == 1), (a == 1) & (b == 0), (a == 1) & (b == 1))):
        place = np.flatnonzero(on)
        place = place[np.lexsort((torque[place], segment[place]))]  # 64 entries: few segments' records, every dof's its own banks
        block = np.stack([segment[place] | torque[place] << 16, place | muscle[place] << 16], 1)
        fill = -len(place) % 64 if kind < 2 else 0
        words += [block, np.tile(np.array([[0, n]], np.int64), (fill, 1))]
        counts.append(len(place) + fill)
    return np.concatenate(words).astype(np.uint32), counts


def _groups_by_kind(kind, columns, fill):
    """Groups ordered by ``kind`` (descending), each kind's filled up to whole wavefronts; (words, kind of every 64)."""
    order = np.argsort(-kind, kind="stable")
    counts = np.bincount(kind, minlength=1)[::-1]
    values = np.flatnonzero(counts)
    counts = counts[values]
    blocks = -(-counts // 64)
    first = 64 * (np.cumsum(blocks) - blocks) - (np.cumsum(counts) - counts)
    at = np.arange(len(kind)) + np.repeat(first, counts)
    out = np.empty((64 * int(blocks.sum()), 4), np.uint32)
    for k in range(4):
        out[:, k] = fill[k]
        out[at, k] = columns[k][order]
    return out, np.repeat(kind.max(initial=0) - values, blocks).astype(np.int32)


def group_context_entries(segment, torque, muscle, start_coeff, end_coeff):
    """The torque's or the gradient's list in groups of up to three entries of one segment and kind (of a list that
    ``pack_context_entries`` takes): (groups (n, 4) uint32, kind | entries << 2 of every 64 groups)."""
    segment, torque, muscle = (np.asarray(a, np.int64) for a in (segment, torque, muscle))
    n = len(segment)
    kind = np.where(np.asarray(start_coeff) == 0, 0, np.where(np.asarray(end_coeff) == 0, 1, 2))
    key = (kind << 16 | segment) << 16 | torque
    order = np.argsort(key)
    key = key[order] >> 16
    run = np.flatnonzero(np.concatenate([[True], key[1:] != key[:-1]]))
    at = np.arange(n) - np.repeat(run, np.diff(np.append(run, n)))  # an entry's number in its segment and kind
    head = np.flatnonzero(at % 3 == 0)
    size = np.diff(np.append(head, n))
    place, dof, key = np.append(order, [n, n]), np.append(torque[order], [0, 0]), key[head]
    p = [place[head], np.where(size > 1, place[head + 1], n), np.where(size > 2, place[head + 2], n)]
    d = [dof[head], np.where(size > 1, dof[head + 1], 0), np.where(size > 2, dof[head + 2], 0)]
    columns = (key & 0xFFFF | d[0] << 16, d[1] | d[2] << 16, muscle[p[0]] | p[0] << 16, p[1] | p[2] << 16)
    return _groups_by_kind(key >> 16 | size << 2, columns, (0, 0, n << 16, n | n << 16))


def group_context_rows(offsets, segment, row_torque, start_coeff, end_coeff):
    """The moment's list with a row's entries, up to three, in a group: (groups (n, 4) uint32, the kinds of every
    64 groups), or None where a row has more or none."""
    offsets, segment, row_torque = (np.asarray(a, np.int64) for a in (offsets, segment, row_torque))
    a, b, n, count = np.asarray(start_coeff), np.asarray(end_coeff), len(segment), np.diff(offsets)
    if count.min(initial=1) < 1 or count.max(initial=0) > 3:
        return None
    kind = np.append(np.where(a == 0, 0, np.where(b == 0, 1, 2)), [3, 3])
    segment, e = np.append(segment, [0, 0]), offsets[:-1]
    seg = [segment[e], np.where(count > 1, segment[e + 1], 0), np.where(count > 2, segment[e + 2], 0)]
    kinds = kind[e] | np.where(count > 1, kind[e + 1], 3) << 2 | np.where(count > 2, kind[e + 2], 3) << 4
    columns = (row_torque | np.arange(len(count)) << 16, seg[0] | seg[1] << 16, seg[2], np.zeros_like(count))
    return _groups_by_kind(kinds, columns, (n << 16, 0, 0, 0))


def _filled(words):
    """Rows of a table up to a multiple of 64, zeros behind them."""
    return np.concatenate([words, np.zeros((-len(words) % 64, words.shape[1]), words.dtype)]).astype(np.uint32).view(np.int32)


class _DeviceTables:
    """Tables of 4-byte words in one allocation on the device, copied there at once: a copy from pageable memory costs the
    same for 100 KB as for one word (24 tables: 0.9 ms)."""

    def __init__(self, device, words: int):
        import torch

        self._host, self._used = np.empty(words, np.int32), 0
        self._device = torch.empty(words, dtype=torch.int32, device=device)

    def add(self, a):
        """The table's place on the device, filled by ``copy``."""
        import torch

        a = np.ascontiguousarray(a)
        if self._used + a.size + 3 > len(self._host):  # (more than was asked for: a copy of its own)
            return torch.from_numpy(a).to(self._device.device)
        at = slice(self._used, self._used + a.size)
        self._host[at] = a.reshape(-1).view(np.int32)
        self._used += (a.size + 3) & ~3
        return self._device[at].view({np.dtype(np.int32): torch.int32, np.dtype(np.float32): torch.float32}[a.dtype]).view(a.shape)

    def copy(self):
        import torch

        self._device[: self._used].copy_(torch.from_numpy(self._host[: self._used]))


def _stream(t) -> int:
    import torch

    return torch.cuda.current_stream(t.device).cuda_stream


class MuscleDynamicsLayer:
    """Static tables of one musculoskeletal model on one GPU and the launchers that use them."""

    def __init__(
        self,
        topology: MuscleTopology,
        *,
        body_count: int,
        full_torque_dim: int,
        torque_dim: int,
        muscle_count: int,
        mechanics: MuscleMechanics | None = None,
        active_torque_indices=None,
        device="cuda",
    ):
        import torch

        if topology.uses_lbs_waypoint_attachments:
            raise NotImplementedError("linear-blend-skinned waypoint attachments are not part of this library")
        if body_count <= 0 or muscle_count <= 0 or torque_dim <= 0:
            raise ValueError("muscle body, muscle, and torque dimensions must be positive")
        if full_torque_dim < torque_dim:
            raise ValueError("full_torque_dim must be at least torque_dim")
        self.mechanics = mechanics or MuscleMechanics()
        self.body_count, self.muscle_count = int(body_count), int(muscle_count)
        self.torque_dim, self.full_torque_dim = int(torque_dim), int(full_torque_dim)
        self.root_dof_count = self.full_torque_dim - self.torque_dim
        self.include_passive_force_in_output = self.mechanics.include_passive_force_in_output
        self.muscle_force_velocity_enabled = False
        self.device = torch.device(device)
        # MuscleOutputSpec.active_torque_indices of the reference (runtime_specs.py:53-63)
        self.active_torque_indices = None if active_torque_indices is None else _np(active_torque_indices)
        self.active_output_dim = self.torque_dim if self.active_torque_indices is None else len(self.active_torque_indices)
        # raw context = xpos | xquat | xipos | subtree_com | cdof (muscle_dynamics.py:4824-4838)
        nb, nvf = self.body_count, self.full_torque_dim
        self._xpos_off, self._xquat_off = 0, 3 * nb
        self._xipos_off, self._com_off, self._cdof_off = 7 * nb, 10 * nb, 13 * nb
        self.context_dim = 13 * nb + 6 * nvf

        t = topology
        self.waypoint_count = len(_np(t.muscle_waypoint_body))
        mask = build_dof_subtree_mask(t.body_parentid, t.dof_bodyid, nb, nvf)
        self.dof_subtree_mask = mask
        body0, body1 = _np(t.apply_segment_body_start_idx), _np(t.apply_segment_body_end_idx)
        self.segment_start_dof_mask = mask[self.root_dof_count :, body0]
        self.segment_end_dof_mask = mask[self.root_dof_count :, body1]
        rootid = _np(t.body_rootid)
        self.apply_segment_muscle_idx = _np(t.apply_segment_muscle_idx, np.int32)
        tq = build_torque_sparse_segment_entries(
            self.segment_start_dof_mask, self.segment_end_dof_mask, t.apply_segment_muscle_idx
        )
        ms = build_muscle_sparse_torque_entries(tq[0], tq[2], tq[4], tq[5], t.apply_segment_muscle_idx, self.muscle_count)
        self.torque_entries_host = tq
        self.muscle_entries_host = ms
        self.sparse_entries: MuscleDofSparseEntries = build_muscle_dof_sparse_entries(
            tq[0], tq[2], tq[3], tq[4], tq[5], self.muscle_count
        )
        self.segments_host = (
            _np(t.apply_segment_start_idx, np.int32), _np(t.apply_segment_end_idx, np.int32),
            rootid[body0].astype(np.int32), rootid[body1].astype(np.int32),
        )  # fmt: skip
        self.all_segment_start_idx = _np(t.all_segment_start_idx, np.int32)
        self.all_muscle_segment_offsets = build_muscle_segment_offsets(t.all_segment_muscle_idx, self.muscle_count)
        self.muscle_params = np.ascontiguousarray(np.asarray(t.muscle_params, np.float32))
        self.muscle_rest_length = np.ascontiguousarray(np.asarray(t.muscle_rest_length, np.float32))
        self.waypoints_local = np.ascontiguousarray(np.asarray(t.muscle_waypoints_local, np.float32))
        self.waypoint_body = _np(t.muscle_waypoint_body, np.int32)
        last = self.all_segment_start_idx.max(initial=-1) + 1
        if max(last, self.segments_host[0].max(initial=-1), self.segments_host[1].max(initial=-1)) >= self.waypoint_count:
            raise ValueError("a segment names a waypoint beyond the waypoint list")
        if self.waypoint_body.max(initial=-1) >= nb or max(self.segments_host[2].max(initial=-1), self.segments_host[3].max(initial=-1)) >= nb:
            raise ValueError("a waypoint or segment names a body beyond body_count")

        m = self.mechanics
        self._model = _lib.MuscleForceModel(
            m.force_scale, m.length_norm_min, m.length_norm_max, (C.c_float * 3)(*m.active_params()),
            (C.c_float * 3)(*m.passive_params()), 1,
        )  # fmt: skip
        self._dev = {}
        if self.device.type == "cuda":
            self._upload()

    # ------------------------------------------------------------------ device tables
    def _upload(self):
        tables = _DeviceTables(self.device, self._table_words())
        up = tables.add
        d = self._dev
        d["seg"] = [up(a) for a in self.segments_host]
        d["tq"] = [up(a) for a in (self.torque_entries_host[i] for i in (0, 2, 3, 4, 5))]
        d["ms"] = [up(a) for a in self.muscle_entries_host]
        e = self.sparse_entries
        d["mom"] = [up(a.astype(np.int32)) for a in (e.muscle_dof_segment_offsets, e.segment_idx)] + [
            up(np.asarray(e.start_coeff, np.float32)),
            up(np.asarray(e.end_coeff, np.float32)),
        ]
        d["mom_torque"] = up(e.muscle_dof_torque_idx.astype(np.int32))
        d["all_seg_start"] = up(self.all_segment_start_idx)
        d["all_seg_off"] = up(self.all_muscle_segment_offsets)
        d["params"], d["rest"] = up(self.muscle_params), up(self.muscle_rest_length)
        d["wp_local"], d["wp_body"] = up(self.waypoints_local), up(self.waypoint_body)
        p = [t.data_ptr() for t in d["seg"]]
        self._segments = _lib.MuscleSegments(*p, len(self.segments_host[0]))

        def entries(ts, nrow, nother, other=True):
            off, seg = ts[0], ts[1]
            rest = ts[2:]
            o = rest[0].data_ptr() if other else None
            a, b = (rest[1], rest[2]) if other else (rest[0], rest[1])
            return _lib.MuscleEntries(off.data_ptr(), seg.data_ptr(), o, a.data_ptr(), b.data_ptr(), nrow, seg.numel(), nother)

        self._torque_entries = entries(d["tq"], self.torque_dim, self.muscle_count)
        self._muscle_entries = entries(d["ms"], self.muscle_count, self.torque_dim)
        self._moment_entries = entries(d["mom"], len(e.muscle_dof_torque_idx), self.torque_dim, other=False)
        self._upload_context(up)
        tables.copy()

    def _table_words(self) -> int:
        """At least the words of all tables, each filled up to 16 bytes."""
        entries, rows, t = len(self.torque_entries_host[2]), len(self.sparse_entries.muscle_dof_torque_idx), self.torque_entries_host
        return 40 * entries + 12 * rows + 12 * self.muscle_count + 8 * self.waypoint_count + 12 * len(self.segments_host[0]) + self.muscle_params.size + 8 * len(t[0]) + 40 * 1024

    def _upload_context(self, up):
        """The argument blocks of im_muscle_from_context, one per output; an output whose entry list or
        sizes it does not take has None and goes by way of waypoints and forces in memory."""
        d, (tq, ms, e) = self._dev, (self.torque_entries_host, self.muscle_entries_host, self.sparse_entries)
        ms_muscle = np.repeat(np.arange(self.muscle_count), np.diff(ms[0]))
        mom_torque = np.repeat(e.muscle_dof_torque_idx, np.diff(e.muscle_dof_segment_offsets))
        lists = (
            (d["tq"][0], self.torque_dim, (tq[2], tq[1], tq[3], tq[4], tq[5])),
            (d["ms"][0], self.muscle_count, (ms[1], ms[2], ms_muscle, ms[3], ms[4])),
            (d["mom"][0], len(e.muscle_dof_torque_idx), (e.segment_idx, mom_torque, np.zeros_like(mom_torque), e.start_coeff, e.end_coeff)),
        )
        self._context = [None, None, None]
        d["packed"] = []
        tables = self._context_tables(up)
        for what, (offsets, nrow, entries) in enumerate(lists):
            packed = pack_context_entries(*entries)
            if packed is None:
                continue
            words, counts = packed
            t = up(words.view(np.int32))
            c = _lib.MuscleContext(
                waypoint_body=d["wp_body"].data_ptr(), waypoint_local=d["wp_local"].data_ptr(),
                all_segment_start=d["all_seg_start"].data_ptr(), all_segment_offsets=d["all_seg_off"].data_ptr(),
                params=d["params"].data_ptr(), rest=d["rest"].data_ptr(), offsets=offsets.data_ptr(), packed=t.data_ptr(),
                ld_params=self.muscle_params.shape[1], nbody=self.body_count, nwaypoint=self.waypoint_count,
                nsegment=len(self.segments_host[0]), ntorque=self.torque_dim, nmuscle=self.muscle_count, nrow=nrow,
                nentry=len(entries[0]), npacked=len(words), kind_count=(C.c_int32 * 3)(*counts), model=self._model,
            )  # fmt: skip
            c.start_waypoint, c.end_waypoint, c.start_root_body, c.end_root_body = (s.data_ptr() for s in d["seg"])
            grouped = (
                group_context_rows(e.muscle_dof_segment_offsets, e.segment_idx, e.muscle_dof_torque_idx, e.start_coeff, e.end_coeff)
                if what == _MOMENT else group_context_entries(*entries)
            )  # fmt: skip
            keep = [t]
            if grouped is not None and tables is not None:
                keep += [up(grouped[0].view(np.int32)), up(grouped[1])]
                c.groups, c.group_kinds = (x.data_ptr() for x in keep[1:])
                c.waypoint_table, c.segment_table, c.length_table, c.muscle_table = (x.data_ptr() for x in tables)
                c.nlength, c.ngroup = len(self.all_segment_start_idx), len(grouped[0])
            if _lib.lib().im_muscle_from_context(C.byref(c), what, None, 0, self.root_dof_count, None, nrow, 0, None) == 0:
                self._context[what] = c
                d["packed"] += keep

    def _context_tables(self, up):
        """The waypoints', segments' and muscles' table entries as im_muscle_from_context loads them beside groups;
        None where a byte offset of a waypoint does not fit 16 bits."""
        if 12 * self.waypoint_count >= 65536 or 12 * self.body_count >= 65536:
            return None
        words = lambda a: np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.int64)  # noqa: E731
        p0, p1, c0, c1 = (12 * a.astype(np.int64) for a in self.segments_host)
        first, count = self.all_muscle_segment_offsets[:-1].astype(np.int64), np.diff(self.all_muscle_segment_offsets)
        zero = np.zeros_like(first)
        tables = (
            np.concatenate([words(self.waypoints_local), 32 * self.waypoint_body[:, None].astype(np.int64)], 1),
            np.stack([p0 | p1 << 16, c0 | c1 << 16], 1), 12 * self.all_segment_start_idx[:, None].astype(np.int64),
            np.stack([first, count, *words(self.muscle_params[:, :3].T), words(self.muscle_rest_length), zero, zero], 1),
        )  # fmt: skip
        self._dev["context_tables"] = [up(_filled(a)) for a in tables]
        return self._dev["context_tables"]

    def _need_gpu(self, *tensors):
        import torch

        if not self._dev:
            raise RuntimeError("this layer was built without a GPU; its kernels exist only in libimhip (no CPU path)")
        for t in tensors:
            if t is None:
                continue
            if not t.is_cuda or t.dtype != torch.float32:
                raise ValueError("muscle tensors must be float32 tensors on the GPU")
            if t.dim() != 2 or (t.numel() and t.shape[1] > 1 and t.stride(1) != 1):
                raise ValueError("muscle tensors must be 2-D with contiguous rows")

    # ------------------------------------------------------------------ geometry
    def _prepare_waypoint_geometry(self, raw_context, *, include_passive_force_magnitude: bool, compute_force_magnitudes: bool = True):
        """Waypoints in the world frame and the per-muscle force magnitudes of a batch of
        contexts (reference _prepare_warp_waypoint_geometry).  Returns a workspace dict and
        the geometry descriptor that the contraction launchers take."""
        import torch

        self._need_gpu(raw_context)
        self._check_context(raw_context)
        B, ld = raw_context.shape[0], raw_context.stride(0)
        base, d, s = raw_context.data_ptr(), self._dev, _stream(raw_context)
        ws = {"transformed_waypoints": torch.empty((B, 3 * self.waypoint_count), device=raw_context.device)}
        wp = ws["transformed_waypoints"]
        L = _lib.lib()
        wp_args = (
            base + 4 * self._xpos_off, ld, base + 4 * self._xquat_off, ld, d["wp_body"].data_ptr(),
            d["wp_local"].data_ptr(), self.waypoint_count, wp.data_ptr(), wp.stride(0),
        )  # fmt: skip
        if compute_force_magnitudes:
            # both steps in one launch: a world's waypoints stay on chip between them
            ws["unit_force_magnitude"] = torch.empty((B, self.muscle_count), device=raw_context.device)
            ws["passive_force_magnitude"] = torch.empty((B, self.muscle_count), device=raw_context.device)
            self._model.include_passive = 1 if include_passive_force_magnitude else 0
            u, p = ws["unit_force_magnitude"], ws["passive_force_magnitude"]
            _lib.check(
                L.im_muscle_waypoints_forces(
                    *wp_args, d["all_seg_start"].data_ptr(), d["all_seg_off"].data_ptr(), d["params"].data_ptr(),
                    self.muscle_params.shape[1], d["rest"].data_ptr(), C.byref(self._model), self.muscle_count,
                    u.data_ptr(), u.stride(0), p.data_ptr(), p.stride(0), B, s,
                ),
                "im_muscle_waypoints_forces",
            )  # fmt: skip
        else:
            _lib.check(L.im_muscle_waypoints(*wp_args, B, s), "im_muscle_waypoints")
        geo = _lib.MuscleGeometry(
            wp.data_ptr(), wp.stride(0), base + 4 * self._com_off, ld, base + 4 * self._cdof_off, ld
        )
        return ws, geo

    def _check_context(self, raw_context):
        """The context's columns; its type, device and rows are ``_need_gpu``'s, which goes before."""
        if raw_context.shape[1] < self.context_dim:
            raise ValueError(f"raw_context has {raw_context.shape[1]} columns, the layer needs {self.context_dim}")

    def _from_context(self, what: int, raw_context, x, out, include_passive_force: bool = False) -> bool:
        """One launch from the context to ``out``, where the layer has a packed list for it."""
        static = self._context[what]
        # (a list that states no range takes the kernels that need none)
        if static is None or not (self._torque_entries, self._muscle_entries, self._moment_entries)[what].nother:
            return False
        c = _lib.MuscleContext.from_buffer_copy(static)  # a call's own block: calls of several threads do not meet
        base, ld = raw_context.data_ptr(), raw_context.stride(0)
        c.xpos, c.xquat = base + 4 * self._xpos_off, base + 4 * self._xquat_off
        c.subtree_com, c.cdof = base + 4 * self._com_off, base + 4 * self._cdof_off
        c.ld_xpos = c.ld_xquat = c.ld_subtree_com = c.ld_cdof = ld
        c.model.include_passive = 1 if include_passive_force else 0
        _lib.check(
            _lib.lib().im_muscle_from_context(
                C.byref(c), what, None if x is None else x.data_ptr(), 0 if x is None else x.stride(0), self.root_dof_count,
                out.data_ptr(), out.stride(0), raw_context.shape[0], _stream(raw_context),
            ),
            "im_muscle_from_context",
        )  # fmt: skip
        return True

    # ------------------------------------------------------------------ launchers
    def _torque_from_context(self, activation, raw_context, include_passive_force: bool):
        """The torque of ``_warp_muscle_dynamics_from_activation_forward`` alone."""
        import torch

        activation, raw_context = activation.float(), raw_context.float()
        self._need_gpu(activation, raw_context)
        if activation.shape != (raw_context.shape[0], self.muscle_count):
            raise ValueError("activation must be (batch, muscle_count)")
        self._check_context(raw_context)
        torque = torch.empty((activation.shape[0], self.torque_dim), device=activation.device)
        if self._from_context(_TORQUE, raw_context, activation, torque, include_passive_force):
            return torque
        return self._warp_muscle_dynamics_from_activation_forward(activation, raw_context, include_passive_force=include_passive_force)[0]

    def _warp_muscle_dynamics_from_activation_forward(self, activation, raw_context, *, include_passive_force: bool, mean_out=None):
        """(torque, transformed_waypoints, unit_force_magnitude), as the reference's method of
        this name (muscle_dynamics.py:4958-5009)."""
        import torch

        activation, raw_context = activation.float(), raw_context.float()
        self._need_gpu(activation, raw_context, mean_out)
        if activation.shape != (raw_context.shape[0], self.muscle_count):
            raise ValueError("activation must be (batch, muscle_count)")
        ws, geo = self._prepare_waypoint_geometry(raw_context, include_passive_force_magnitude=include_passive_force)
        B = activation.shape[0]
        mean = mean_out if mean_out is not None else torch.empty((B, self.torque_dim), device=activation.device)
        u, p = ws["unit_force_magnitude"], ws["passive_force_magnitude"]
        _lib.check(
            _lib.lib().im_muscle_torque_forward(
                C.byref(geo), C.byref(self._segments), C.byref(self._torque_entries), u.data_ptr(), u.stride(0),
                p.data_ptr() if include_passive_force else None, p.stride(0), activation.data_ptr(),
                activation.stride(0), self.root_dof_count, mean.data_ptr(), mean.stride(0), B, _stream(activation),
            ),
            "im_muscle_torque_forward",
        )  # fmt: skip
        return mean, ws["transformed_waypoints"], u

    def _warp_muscle_dynamics_from_activation_backward(self, raw_context, grad_output, unit_force_magnitude=None):
        """Activation gradient; geometry is rebuilt from the context unless the unit forces
        are handed in."""
        import torch

        raw_context, grad_output = raw_context.float(), grad_output.float().contiguous()
        self._need_gpu(raw_context, grad_output, unit_force_magnitude)
        if grad_output.shape != (raw_context.shape[0], self.torque_dim):
            raise ValueError("grad_output must be (batch, torque_dim)")
        if unit_force_magnitude is None:
            self._check_context(raw_context)
            grad = torch.empty((raw_context.shape[0], self.muscle_count), device=raw_context.device)
            if self._from_context(_GRAD, raw_context, grad_output, grad):
                return grad
        ws, geo = self._prepare_waypoint_geometry(
            raw_context, include_passive_force_magnitude=False, compute_force_magnitudes=unit_force_magnitude is None
        )
        u = ws["unit_force_magnitude"] if unit_force_magnitude is None else unit_force_magnitude
        B = raw_context.shape[0]
        grad = torch.empty((B, self.muscle_count), device=raw_context.device)
        _lib.check(
            _lib.lib().im_muscle_activation_grad(
                C.byref(geo), C.byref(self._segments), C.byref(self._muscle_entries), u.data_ptr(), u.stride(0),
                grad_output.data_ptr(), grad_output.stride(0), self.root_dof_count, grad.data_ptr(), grad.stride(0), B,
                _stream(raw_context),
            ),
            "im_muscle_activation_grad",
        )  # fmt: skip
        return grad

    def _warp_muscle_dynamics_from_activation_forward_cached_lbs_force(
        self, activation, raw_context, unit_force_magnitude, passive_force_magnitude, *, include_passive_force: bool
    ):
        """Torque from force magnitudes computed outside this call (the reference method of
        this name behind instantmimic_muscle::torque_cached_lbs_forward)."""
        import torch

        activation, raw_context = activation.float(), raw_context.float()
        self._need_gpu(activation, raw_context, unit_force_magnitude, passive_force_magnitude)
        B = activation.shape[0]
        for t in (activation, unit_force_magnitude, passive_force_magnitude):
            if tuple(t.shape) != (B, self.muscle_count):
                raise ValueError("activation and force magnitudes must be (batch, muscle_count)")
        _, geo = self._prepare_waypoint_geometry(raw_context, include_passive_force_magnitude=False, compute_force_magnitudes=False)
        mean = torch.empty((B, self.torque_dim), device=activation.device)
        u, p = unit_force_magnitude, passive_force_magnitude
        _lib.check(
            _lib.lib().im_muscle_torque_forward(
                C.byref(geo), C.byref(self._segments), C.byref(self._torque_entries), u.data_ptr(), u.stride(0),
                p.data_ptr() if include_passive_force else None, p.stride(0), activation.data_ptr(),
                activation.stride(0), self.root_dof_count, mean.data_ptr(), mean.stride(0), B, _stream(activation),
            ),
            "im_muscle_torque_forward",
        )  # fmt: skip
        return mean

    def _compute_activation_torque_bounds_warp(self, raw_context, *, select_active: bool):
        """(lower, upper) of the torque over activations in [0, 1] at the context's geometry
        (reference muscle_dynamics.py:4810-4822); ``select_active`` keeps the layer's
        active torque indices."""
        import torch

        raw_context = raw_context.float()
        self._need_gpu(raw_context)
        ws, geo = self._prepare_waypoint_geometry(raw_context, include_passive_force_magnitude=False)
        B = raw_context.shape[0]
        lower = torch.empty((B, self.torque_dim), device=raw_context.device)
        upper = torch.empty_like(lower)
        u = ws["unit_force_magnitude"]
        _lib.check(
            _lib.lib().im_muscle_torque_bounds(
                C.byref(geo), C.byref(self._segments), C.byref(self._torque_entries), u.data_ptr(), u.stride(0),
                self.root_dof_count, lower.data_ptr(), upper.data_ptr(), lower.stride(0), B, _stream(raw_context),
            ),
            "im_muscle_torque_bounds",
        )  # fmt: skip
        if select_active and self.active_torque_indices is not None:
            idx = torch.from_numpy(self.active_torque_indices.astype(np.int64)).to(raw_context.device)
            return lower.index_select(1, idx), upper.index_select(1, idx)
        return lower, upper

    def eval_muscle_sparse_moment(self, raw_context, moment_out=None):
        """moment (batch, entries) of the (muscle, dof) entries in ``sparse_entries``
        (reference eval_muscle_sparse_moment_kernel, muscle_qfrc_projector.py:2617-2662)."""
        import torch

        raw_context = raw_context.float()
        self._need_gpu(raw_context, moment_out)
        self._check_context(raw_context)
        if moment_out is None:
            moment_out = torch.empty((raw_context.shape[0], len(self.sparse_entries.muscle_dof_torque_idx)), device=raw_context.device)
        if self._from_context(_MOMENT, raw_context, None, moment_out):
            return moment_out
        ws, geo = self._prepare_waypoint_geometry(raw_context, include_passive_force_magnitude=False, compute_force_magnitudes=False)
        B, moment = raw_context.shape[0], moment_out
        _lib.check(
            _lib.lib().im_muscle_sparse_moment(
                C.byref(geo), C.byref(self._segments), self._dev["mom_torque"].data_ptr(), C.byref(self._moment_entries),
                self.root_dof_count, moment.data_ptr(), moment.stride(0), B, _stream(raw_context),
            ),
            "im_muscle_sparse_moment",
        )  # fmt: skip
        return moment

    def forward_from_activation(self, activation, raw_context, include_passive_force: bool | None = None):
        """Differentiable torque through the dispatcher operator."""
        from .warp_custom_ops import muscle_torque_forward, warp_op_key

        inc = self.include_passive_force_in_output if include_passive_force is None else bool(include_passive_force)
        return muscle_torque_forward(activation, raw_context, warp_op_key(self), inc)
