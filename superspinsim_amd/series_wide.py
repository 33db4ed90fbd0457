"""The series in the drive for models of 65 to 192 states
(``ssmx_propagate_series_wide``): matrices, layout and launch.

The E_k of a model this size are sparse where its couplings are nearly
block-diagonal (a nucleus on a spin: 171 states, about 70 significant entries
a row).  Entries whose sum over a column, at the run's largest drive, stays
below a share of the tolerance are left out; what remains is laid out as row
pairs over 8 or 16 lanes each.
"""

import ctypes
import math

import numpy as np

from superspinsim_amd import _lib
from superspinsim_amd.propagator import (
    _ptr, _torch, device_tensor, record_use)
from superspinsim_amd.series import (
    ORDERS, _dropped, chebyshev, economised, split_sectors)

_f64 = np.float64

#: the kernel's limits: rows (eight pairs in each wavefront), wavefronts,
#: columns per lane
MAX_ROWS, MAX_WAVES, MIN_SLOTS, MAX_SLOTS = 192, 12, 4, 8
#: rows of a model beyond which none is built (up to here it has no plan)
MAX_STATES = 256
#: highest 1-norm of h w C (beyond, the E_k fill in past the kernel's limits)
MAX_NORM = 1.0
#: highest order computed for the first of ORDERS, and for the others
TOP = (4, 6)
#: columns per lane whose orders 0..3 registers hold; KB of LDS for the other
#: coefficients (one KB per column and order, for both rows of the pairs)
REG_SLOTS, LDS_COLUMNS = 7, 150
#: share of the tolerance that left-out entries may take, per column
SHARE = 1.0 / 64.0


def wide_coefficients(terms, drive, orders):
    """``coefficient_matrices`` where the extended products of every term
    take a second (171 states): those up to a degree d are summed in extended
    precision, the others in doubles.

    For a constant part of 1-norm c the terms beyond degree d are
    c^d / (d + 1)! of it; d is the first where that is below 1/96 (2 for
    c <= 1/4), so that their rounding (some 10 ulp) stays a tenth of the
    rounding of the result.
    """
    const = sum(np.asarray(m, dtype=np.longdouble) * np.longdouble(s)
                for m, s in terms)
    n = const.shape[0]
    norm = float(np.abs(const).sum(axis=0).max(initial=0.0))
    drive = np.asarray(drive, dtype=_f64)
    exact, size = 2, norm ** 2 / 6.0
    while size > 1.0 / 96.0:
        exact += 1
        size *= norm / (exact + 1)

    def lists(mat):
        return [(c, mat[r, c]) for r, c in
                ((r, np.flatnonzero(mat[r])) for r in range(n))]

    def times(rows, mat):
        return np.stack([v @ mat[c] for c, v in rows])

    rows, drows = lists(const), lists(drive)
    # orders above the degree are zero
    term = [const, drive.astype(np.longdouble)][:orders + 1]
    total = list(term)
    for t in range(2, exact + 1):
        new = [times(rows, m) for m in term]
        for k, m in enumerate(term[:orders]):
            v = times(drows, m)
            if k + 1 < len(new):
                new[k + 1] += v
            else:
                new.append(v)
        term = [m / t for m in new]
        total = [m + term[k] if k < len(total) else term[k]
                 for k, m in enumerate(total + term[len(total):])]
    last = np.zeros((orders + 1, n, n))
    for k, m in enumerate(term):
        last[k] = m
    small = np.zeros((orders + 1, n, n))
    c64 = const.astype(_f64)
    bound, t = 1.0, exact
    while bound > 1e-18 or t <= orders + 2:
        t += 1
        # an order's terms go like norm^(t - k) / (t - k)! of its first
        bound = norm ** max(t - orders, 0) / math.factorial(
            max(t - orders, 0))
        new = c64 @ last
        new[1:] += drive @ last[:-1]
        last = new / t
        small += last
    return [(total[k] + small[k] if k < len(total) else
             small[k].astype(np.longdouble)).astype(_f64)
            for k in range(orders + 1)]


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
    """E_k of one (constant, drive) pair of 65..192 states at one step size;
    ``build`` or ``plan`` returns None where the kernel does not apply."""

    def __init__(self):
        self._layout = None         # the last drive's

    @classmethod
    def build(cls, const, drive, weights, h):
        n = const.shape[0]
        sums = weights.sum(axis=1)
        if not _lib.MAX_N < n <= MAX_STATES or weights.shape != (2, 2) or \
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
        self.mats = []
        self._point = terms, drive
        self.drive_norm = float(np.abs(drive).sum(axis=0).max())
        return self

    def plan(self, drive_max, tol):
        """(da, db, F, budget) for drives |c(t)| <= ``drive_max``, or None;
        the bound of ``SeriesModel.plan`` with the left-out entries added."""
        if self.n > MAX_ROWS:
            return None
        F = self.h * self.weight * float(drive_max)
        budget = SHARE * tol
        # (drives that the first orders may not do for: all at once)
        b = F * self.drive_norm
        small = b <= 1.0 and b ** 4 / 24.0 <= tol
        for da, db in ORDERS:
            top = TOP[0] if small and (da, db) == ORDERS[0] else TOP[1]
            mats = self.mats
            if len(mats) <= top:
                mats = wide_coefficients(*self._point, top)
                # (a thread with a larger drive may have kept more)
                if len(mats) > len(self.mats):
                    self.mats = mats
            worst = [np.abs(c).sum(axis=0).max() for c in chebyshev(mats, F)]
            if not np.all(np.isfinite(worst)):
                return None
            if 8.0 * (budget + worst[-1] + sum(
                    worst[k] for k in _dropped(len(worst), da, db))) <= tol:
                plan = da, db, F, budget
                return None if self.layout(plan) is None else plan
        return None

    def flops(self, plan):
        """FP64 operations of one exponential: a multiply-add per order and
        kept entry, two per row."""
        even, odd = self.entries
        return int(2 * (even * (plan[0] + 1) + odd * (plan[1] + 1) +
                        2 * self.n))

    def layout(self, plan):
        """(blocks, states, columns, table) of the kernel, on the device but
        for the states, and its columns in LDS; None where the rows don't
        fit it."""
        # (another thread may keep its own drive's in between)
        kept = self._layout
        if kept is None or kept[0] != plan:
            self._layout = kept = plan, self._staged(self._arrays(*plan))
        return kept[1]

    def transposed(self, plan):
        """``layout`` of the transposed matrices (not kept)."""
        return self._staged(self._arrays(*plan, transpose=True))

    @staticmethod
    def _staged(arrays):
        if arrays is None:
            return None
        blocks, states, columns, table, in_lds = arrays
        return device_tensor(blocks), states, device_tensor(columns), \
            device_tensor(table), in_lds

    def _arrays(self, da, db, F, budget, transpose=False):
        kept = economised(self.mats, da, db, F)
        kept = [kept[k] for k in range(2 * max(da, db) + 2)
                if k <= (2 * db + 1 if k % 2 else 2 * da)]
        if transpose:
            kept = [np.ascontiguousarray(m.T) for m in kept]
        size = sum(F ** k * np.abs(m) for k, m in enumerate(kept))
        order = np.argsort(size, axis=0, kind="stable")
        keep = np.empty(size.shape, dtype=bool)
        np.put_along_axis(keep, order, np.cumsum(np.take_along_axis(
            size, order, axis=0), axis=0) >= budget, axis=0)
        same = self.sector[:, None] == self.sector[None, :]
        self.entries = (np.count_nonzero(keep & same),
                        np.count_nonzero(keep & ~same))
        pairs = pair_rows(keep, self.sector)
        cols = []
        for a, b in pairs:
            union = keep[a] | keep[b] if b >= 0 else keep[a]
            cols.append((np.flatnonzero(union & same[a]),
                         np.flatnonzero(union & ~same[a])))
        widest = np.array([max(o.size, p.size) for o, p in cols])
        rank = np.argsort(-widest, kind="stable")
        waves = self._waves(widest[rank])
        # orders above 3 and columns beyond the registers' lie in LDS
        high = da - 1 + db - 1
        if waves is None:
            return None
        in_lds = sum(high * s + 4 * max(0, s - REG_SLOTS) for _, s in waves)
        if in_lds > LDS_COLUMNS:
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
            hi = np.zeros((high, slots, 64, 2))
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
                        if r < 0:
                            continue
                        use = keep[r, cols[p][part]]
                        for o in (0, 1):
                            t[slot, 2 * o + i, lane] = \
                                kept[2 * o + part][r, cols[p][part]] * use
                        if high > part:
                            hi[part, e // lanes, lane, i] = \
                                kept[4 + part][r, cols[p][part]] * use
            first += 64 // lanes
            done += c.size
            parts = [t[:slots][:REG_SLOTS], t[slots:][:REG_SLOTS], hi]
            if slots > REG_SLOTS:
                # [column][own 0, 2, opposite 1, 3][lane][row]
                rest = np.stack([t[REG_SLOTS:slots],
                                 t[slots + REG_SLOTS:]], axis=1)
                parts.append(rest.reshape(-1, 2, 2, 2, 64).transpose(
                    0, 1, 2, 4, 3))
            columns.append(c.ravel())
            table += [part.ravel() for part in parts]
            tabled += sum(part.size for part in parts)
        return blocks, states, np.concatenate(columns), \
            np.concatenate(table), in_lds

    @staticmethod
    def _waves(widest):
        """[(lanes per pair, columns per lane)] of the wavefronts for pairs
        sorted by width: as few 16-lane ones as leave the others within the
        registers' columns per lane, or else within the kernel's."""
        for most in (REG_SLOTS, MAX_SLOTS):
            for wide in range(MAX_WAVES + 1):
                out, i = [], 0
                while i < widest.size:
                    lanes = 16 if len(out) < wide else 8
                    slots = -(-int(widest[i]) // lanes)
                    out.append((lanes, max(slots, MIN_SLOTS)))
                    i += 64 // lanes
                if len(out) <= MAX_WAVES and \
                        max(s for _, s in out) <= most:
                    return out
        return None


def own_states(lane_states, states):
    """``lane_states`` of a layout with the caller's state indices."""
    out = lane_states.copy()
    out[..., 1] = np.asarray(states)[lane_states[..., 1]]
    return out


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
        self.blocks, lane_states, self.columns, self.table, in_lds = \
            model.layout(plan)
        self.states = device_tensor(own_states(lane_states, states))
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
            lds_columns=in_lds, da=plan[0], db=plan[1], h=dt / fine, t0=t0,
            dt=dt)
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
        # (shared by the model's runs)
        record_use(self.blocks, self.columns, self.table)
        return self.out

    def result(self):
        return self.out
