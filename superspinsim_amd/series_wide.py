"""The series in the drive for models of 65 to 256 states
(``ssmx_propagate_series_wide``): matrices, layout and launch.

The E_k of a model this size are sparse where its couplings are nearly
block-diagonal (a nucleus on a spin: 171 states, about 70 significant entries
a row).  Entries whose sum over a column, at the run's largest drive, stays
below a share of the tolerance are left out; what remains is laid out as row
pairs over 8 or 16 lanes each.
"""

import ctypes

import numpy as np

from superspinsim_amd import _lib
from superspinsim_amd.propagator import _ptr, _torch, device_tensor
from superspinsim_amd.series import (
    MAX_NORM, SeriesModel, _dropped, coefficient_matrices, split_sectors)

_f64 = np.float64

#: the kernel's limits: rows, wavefronts, columns per lane
MAX_ROWS, MAX_WAVES, MIN_SLOTS, MAX_SLOTS = 256, 12, 4, 7
#: orders kept (even 0, 2; odd 1, 3) and computed, which bounds the rest
DA, DB, TOP = 1, 1, 4
#: share of the tolerance that left-out entries may take, per column
SHARE = 1.0 / 64.0


def wide_coefficients(terms, drive, orders):
    """``coefficient_matrices`` where the extended products of every term
    take a second (171 states): those of degree one and two are summed in
    extended precision, the others in doubles.

    For a constant part of 1-norm c <= 1/4 the terms from degree three on
    are c^3 / 6 of it, so that their rounding (some 10 ulp) stays a tenth of
    the rounding of the result.  Larger ones take the extended products.
    """
    const = sum(np.asarray(m, dtype=np.longdouble) * np.longdouble(s)
                for m, s in terms)
    n = const.shape[0]
    norm = float(np.abs(const).sum(axis=0).max(initial=0.0))
    if not norm <= 0.25:
        return coefficient_matrices(terms, drive, orders)
    drive = np.asarray(drive, dtype=_f64)
    rows = [(c, const[r, c]) for r, c in
            ((r, np.flatnonzero(const[r])) for r in range(n))]
    drows = [(c, drive[r, c]) for r, c in
             ((r, np.flatnonzero(drive[r])) for r in range(n))]

    def times(lists, mat):
        return np.stack([v @ mat[c] for c, v in lists])

    first = [const, drive.astype(np.longdouble)]
    half = np.longdouble(0.5)
    second = [times(rows, const) * half,
              (times(drows, const) + times(rows, first[1])) * half,
              times(drows, first[1]) * half]
    zero = np.zeros((n, n), dtype=np.longdouble)
    total = [(first + [zero] * orders)[k] + (second + [zero] * orders)[k]
             for k in range(orders + 1)]
    term = np.zeros((orders + 1, n, n))
    for k in range(min(orders, 2) + 1):
        term[k] = second[k]
    small = np.zeros((orders + 1, n, n))
    c64 = const.astype(_f64)
    bound, t = 1.0, 2
    while bound > 1e-24 or t <= orders + 2:
        t += 1
        bound *= norm / max(t - orders, 1)
        new = c64 @ term
        new[1:] += drive @ term[:-1]
        term = new / t
        small += term
    return [(m + s).astype(_f64) for m, s in zip(total, small)]


def pair_rows(pattern, sector):
    """Pairs of rows (second -1: none) of one sector whose columns overlap
    most: best matches first, the wider ones among equals."""
    n = pattern.shape[0]
    p = pattern.astype(_f64)
    common, size = p @ p.T, p.sum(axis=1)
    a, b = np.triu_indices(n, 1)
    same = sector[a] == sector[b]
    a, b = a[same], b[same]
    widest = np.maximum(np.maximum(size[a], size[b]), 1.0)
    score = (size[a] + size[b] - common[a, b]) / widest - 1e-3 * widest
    free = np.ones(n, dtype=bool)
    pairs = []
    for i in np.argsort(score, kind="stable"):
        if free[a[i]] and free[b[i]]:
            free[a[i]] = free[b[i]] = False
            pairs.append((int(a[i]), int(b[i])))
    return pairs + [(int(r), -1) for r in np.flatnonzero(free)]


class WideModel:
    """E_k of one (constant, drive) pair of 65..256 states at one step size;
    ``build`` returns None where the kernel does not apply."""

    def __init__(self):
        self._layout = None         # the last drive's

    @classmethod
    def build(cls, const, drive, weights, h):
        n = const.shape[0]
        sums = weights.sum(axis=1)
        if not _lib.MAX_N < n <= MAX_ROWS or weights.shape != (2, 2) or \
                not np.allclose(sums[0], sums[1], rtol=1e-15, atol=1e-16):
            return None
        terms = [(const, h * float(sums[0]))]
        if not abs(terms[0][1]) * np.abs(const).sum(axis=0).max() <= MAX_NORM:
            return None
        found = split_sectors(const, drive)
        if found is None:
            return None
        self = cls()
        self.n, self.h = n, h
        self.sector = found[0]
        # LDS rows by sector: the lanes of a pair then read runs of
        # neighbours, and pairs with common columns the same ones
        self.pos = np.empty(n, dtype=np.int32)
        self.pos[np.argsort(self.sector, kind="stable")] = np.arange(n)
        self.size = int(np.bincount(self.sector).max())
        self.weight = float(np.abs(weights).sum(axis=1).max())
        self.nnz = int(np.count_nonzero((const != 0) | (drive != 0)))
        self.mats = wide_coefficients(terms, drive, TOP)
        return self

    def plan(self, drive_max, tol):
        """(da, db, F, budget) for drives |c(t)| <= ``drive_max``, or None;
        the bound of ``SeriesModel.plan`` with the left-out entries added."""
        F = self.h * self.weight * float(drive_max)
        worst = [np.abs(c).sum(axis=0).max()
                 for c in SeriesModel._chebyshev(self.mats, F)]
        if not np.all(np.isfinite(worst)):
            return None
        budget = SHARE * tol
        if not 8.0 * (budget + worst[-1] + sum(
                worst[k] for k in _dropped(TOP + 1, DA, DB))) <= tol:
            return None
        plan = DA, DB, F, budget
        return None if self.layout(plan) is None else plan

    def layout(self, plan):
        """Device (blocks, states, columns, table) of the kernel, or None
        where the rows don't fit it."""
        if self._layout is None or self._layout[0] != plan:
            arrays = self._arrays(*plan[2:])
            self._layout = (plan, None if arrays is None else
                            tuple(device_tensor(a) for a in arrays))
        return self._layout[1]

    def transposed(self, plan):
        """``layout`` of the transposed matrices, on the host."""
        return self._arrays(*plan[2:], transpose=True)

    def _arrays(self, F, budget, transpose=False):
        kept = [m.copy() for m in self.mats[:4]]
        # the dropped order's Chebyshev polynomial taken off
        # (T_4 = 8 u^4 - 8 u^2 + 1: its lower coefficients stay with E_0, E_2)
        top = F ** 4 / 8.0 * self.mats[4]
        if F ** 2 > 0.0:
            kept[0] -= top
            kept[2] += (8.0 / F ** 2) * top
        if transpose:
            kept = [np.ascontiguousarray(m.T) for m in kept]
        size = sum(F ** k * np.abs(m) for k, m in enumerate(kept))
        order = np.argsort(size, axis=0, kind="stable")
        keep = np.empty(size.shape, dtype=bool)
        np.put_along_axis(keep, order, np.cumsum(np.take_along_axis(
            size, order, axis=0), axis=0) >= budget, axis=0)
        same = self.sector[:, None] == self.sector[None, :]
        pairs = pair_rows(keep, self.sector)
        cols = []
        for a, b in pairs:
            union = keep[a] | keep[b] if b >= 0 else keep[a]
            cols.append((np.flatnonzero(union & same[a]),
                         np.flatnonzero(union & ~same[a])))
        widest = np.array([max(o.size, p.size) for o, p in cols])
        rank = np.argsort(-widest, kind="stable")
        waves = self._waves(widest[rank])
        if waves is None:
            return None
        pos = self.pos
        blocks = np.zeros((len(waves), 4), dtype=np.int32)
        states = np.zeros((len(waves), 64, 2), dtype=np.int32)
        states[:, :, 0] = -1
        columns, table = [], []
        first = done = tabled = 0
        for w, (lanes, slots) in enumerate(waves):
            blocks[w] = slots, lanes, done, tabled
            c = np.zeros((2 * slots, 64), dtype=np.int32)
            t = np.zeros((2 * slots, 4, 64))
            for g in range(64 // lanes):
                if first + g >= len(pairs):
                    break
                p = rank[first + g]
                h = lanes // 2
                mine = 32 * np.arange(2)[:, None] + g * h + np.arange(h)
                c[:, mine.ravel()] = pos[pairs[p][0]]
                for i, r in enumerate(pairs[p]):
                    if r < 0:
                        continue
                    states[w, mine[i], 0], states[w, mine[i], 1] = pos[r], r
                for part in (0, 1):
                    e = np.arange(cols[p][part].size)
                    slot = part * slots + e // lanes
                    lane = mine.ravel()[e % lanes]
                    c[slot, lane] = pos[cols[p][part]]
                    for i, r in enumerate(pairs[p]):
                        for o in (0, 1):
                            if r >= 0:
                                t[slot, 2 * o + i, lane] = \
                                    kept[2 * o + part][r, cols[p][part]] * \
                                    keep[r, cols[p][part]]
            first += 64 // lanes
            done += c.size
            tabled += t.size
            columns.append(c.ravel())
            table.append(t.ravel())
        return blocks, states, np.concatenate(columns), np.concatenate(table)

    @staticmethod
    def _waves(widest):
        """[(lanes per pair, columns per lane)] of the wavefronts for pairs
        sorted by width: as few 16-lane ones as leave the others within
        the kernel's columns per lane."""
        for wide in range(MAX_WAVES + 1):
            out, i = [], 0
            while i < widest.size:
                lanes = 16 if len(out) < wide else 8
                slots = -(-int(widest[i]) // lanes)
                out.append((lanes, max(slots, MIN_SLOTS)))
                i += 64 // lanes
            if len(out) <= MAX_WAVES and max(s for _, s in out) <= MAX_SLOTS:
                return out
        return None


class WideRun:
    """Staged inputs of one run through ``ssmx_propagate_series_wide``;
    arguments as ``SeriesRun``."""

    k = 1

    def __init__(self, model, plan, states, weights, nodes, rho0, d_waves,
                 d_segs, gen, fine, n_out, t0, dt, obs, read):
        torch = _torch()
        n_inst, n = rho0.shape
        flags = {"full": _lib.SSMX_READ_FULL, "obs": 0,
                 "integral": _lib.SSMX_READ_INTEGRAL}[read]
        n_obs = obs.shape[0] if obs is not None and read != "full" else 0
        if read != "full" and not 1 <= n_obs <= _lib.MAX_OBS:
            raise ValueError(f"{n_obs} readout rows outside 1.."
                             f"{_lib.MAX_OBS}")
        self.blocks, lane_states, self.columns, self.table = \
            model.layout(plan)
        # the kernel's state index is the caller's
        index = device_tensor(np.asarray(states).astype(np.int32))
        self.states = torch.stack(
            [lane_states[..., 0], index[lane_states[..., 1].long()]], dim=-1)
        self.d_w, self.d_nodes = device_tensor(weights), device_tensor(nodes)
        self.d_rho0, self.d_waves, self.d_segs = (
            device_tensor(np.ascontiguousarray(rho0, dtype=_f64)), d_waves,
            d_segs)
        self.d_obs = None if read == "full" else device_tensor(
            np.ascontiguousarray(obs, dtype=_f64))
        self.partial = model.n < n
        self.desc = _lib.SeriesDesc(
            n=n, rows=model.n, n_inst=n_inst, members=1,
            n_exp=weights.shape[0], n_node=weights.shape[1], fine=fine,
            n_out=n_out, n_obs=n_obs, flags=flags, gen=gen, wave_group=1,
            da=plan[0], db=plan[1], h=dt / fine, t0=t0, dt=dt)
        shape = {"full": (n_inst, n_out, n), "obs": (n_inst, n_out, n_obs),
                 "integral": (n_inst, n_obs)}[read]
        self.out = torch.empty(shape, dtype=torch.float64, device="cuda")

    def launch(self):
        if self.partial and self.desc.flags & _lib.SSMX_READ_FULL:
            self.out.zero_()
        _lib.check(_lib.load().ssmx_propagate_series_wide(
            ctypes.byref(self.desc), _ptr(self.blocks),
            self.blocks.shape[0], _ptr(self.states), _ptr(self.columns),
            _ptr(self.table), _ptr(self.d_w), _ptr(self.d_nodes),
            _ptr(self.d_waves), _ptr(self.d_segs), _ptr(self.d_rho0),
            _ptr(self.d_obs), _ptr(self.out), None, None, ctypes.c_void_p(
                _torch().cuda.current_stream().cuda_stream)))
        return self.out

    def result(self):
        return self.out
