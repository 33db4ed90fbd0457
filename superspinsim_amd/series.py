"""Series-in-the-drive tables: plan and launch of ``ssmx_propagate_series``.

An exponent ``h w C + f G`` with a constant matrix C and one driven matrix G
is exponentiated as ``I + sum_k f^k E_k``, where ``E_k`` collects every term
of order k in G (``coefficient_matrices``).  For the drives of magnetic
resonance f G is small (1-norm about 1e-3 at 20 ps steps), so four or five
orders reach the accuracy that takes a Taylor chain in the whole exponent
11 products.

``reachable`` finds the states a run can involve at all: those that the
couplings connect to the initial states and to the readout.  The others stay
exactly zero or are never read (a sweep that starts from populations never
fills the coherences between the orbital blocks).
"""

import ctypes
import math

import numpy as np

from superspinsim_amd import _lib
from superspinsim_amd.propagator import (
    _ptr, _torch, device_tensor, record_use)

_f64 = np.float64

def simd_count():
    """SIMDs of the device (four per CU)."""
    return 4 * _torch().cuda.get_device_properties(0).multi_processor_count


#: components per sector the kernels hold
SIZES = (5, 11)
#: (highest even order / 2, (highest odd order - 1) / 2), cheapest first
ORDERS = ((1, 1), (2, 1), (2, 2))
#: highest 1-norm of h w C (the series of E_0 then loses under one digit)
MAX_NORM = 4.0


def reachable(pattern, rho0, obs=None):
    """Indices of the states a run can involve.

    ``pattern[a, b]`` is set where some generator takes state b to state a;
    ``rho0`` (instances, n) are the initial states.  States that no non-zero
    initial component reaches stay zero; with readout rows ``obs`` those
    that no read component depends on are left out as well.
    """
    def closure(adjacency, start):
        seen = start.copy()
        front = start
        while front.any():
            front = adjacency[:, front].any(axis=1) & ~seen
            seen |= front
        return seen

    # a NaN or an infinite component counts as filled
    keep = closure(pattern, np.any(rho0 != 0, axis=0))
    if obs is not None:
        keep &= closure(pattern.T, np.any(obs != 0, axis=0))
    return np.flatnonzero(keep)


class Reach:
    """States that gradients involve: what the run reaches from ``rho0`` and
    what the readout ``obs`` depends on (a parameter may join one to the
    other)."""

    def __init__(self, pattern, rho0, obs):
        n = pattern.shape[0]
        self.ahead, self.behind = np.zeros((2, n), dtype=bool)
        self.ahead[reachable(pattern, rho0)] = True
        self.behind[reachable(pattern.T, obs)] = True
        self.states = np.flatnonzero(self.ahead | self.behind)

    def covers(self, obs, rho0=None):
        """Whether other rows (and initial states) involve no further
        ones."""
        def within(rows, mask):
            return rows.shape[-1] == mask.size and \
                not np.any(rows[:, ~mask] != 0)

        return within(obs, self.behind) and \
            (rho0 is None or within(rho0, self.ahead))


def split_sectors(const, drive):
    """(sector of each state, opposite sector of each sector) or None.

    Sectors are the groups that ``const`` couples (in either direction);
    ``drive`` must couple every state of a sector to states of one other
    sector only, and that one back to it.  Sectors that the drive leaves
    alone are their own opposite's empty partner (-1).
    """
    n = const.shape[0]
    even = (const != 0) | (const.T != 0)
    odd = (drive != 0) | (drive.T != 0)
    # two-colour the connected components: even edges keep the colour, odd
    # edges change it
    comp = np.full(n, -1)
    colour = np.zeros(n, dtype=np.int64)
    count = 0
    for s in range(n):
        if comp[s] >= 0:
            continue
        comp[s], stack = count, [s]
        while stack:
            a = stack.pop()
            for b in np.flatnonzero((even[a] | odd[a]) & (comp < 0)):
                if even[a, b] and odd[a, b]:
                    return None
                comp[b] = count
                colour[b] = colour[a] ^ int(odd[a, b])
                stack.append(b)
        count += 1
    same = comp[:, None] == comp[None, :]
    flip = colour[:, None] != colour[None, :]
    if np.any(even & same & flip) or np.any(odd & ~flip):
        return None
    sector = 2 * comp + colour
    names, sector = np.unique(sector, return_inverse=True)
    index = {int(v): k for k, v in enumerate(names)}
    opposite = np.array([index.get(int(v) ^ 1, -1) for v in names])
    return sector, opposite


def _dropped(count, da, db):
    """Orders below ``count`` that the kernels' (da, db) leave out."""
    return [k for k in range(count)
            if k > (2 * da if k % 2 == 0 else 2 * db + 1)]


def _sparse(mats):
    """(columns, values [..., slot, row]), slot by slot, of the rows of
    ``mats`` (..., n, n) over their common pattern."""
    n = mats.shape[-1]
    pattern = np.any(mats.reshape(-1, n, n) != 0, axis=0)
    width = int(np.max(np.count_nonzero(pattern, axis=1), initial=0))
    cols = np.zeros((width, n), dtype=np.int64)
    vals = np.zeros(mats.shape[:-2] + (width, n), dtype=np.longdouble)
    for r in range(n):
        c = np.flatnonzero(pattern[r])
        cols[:c.size, r] = c
        vals[..., :c.size, r] = mats[..., r, c]
    return cols, vals


def coefficient_stacks(sets, drive, orders, extended=False):
    """``coefficient_matrices`` of every element of ``sets`` (terms) at once:
    per order one array (sets, n, n).

    A set's values are those it has alone; together they take half as long
    as one by one (19 states)."""
    const = np.stack([sum(np.asarray(m, dtype=np.longdouble) *
                          np.longdouble(s) for m, s in terms)
                      for terms in sets])
    n = const.shape[-1]
    cc, cv = _sparse(const)
    dc, dv = _sparse(np.asarray(drive, dtype=_f64))

    def times(cols, vals, mat):
        out = np.zeros_like(mat)
        for k, c in enumerate(cols):
            part = mat.take(c, axis=1)
            part *= vals[..., k, :, None]
            out += part
        return out

    # terms of order t in const fall like norm^t / t!, drive orders add to t
    count = np.zeros(len(sets), dtype=np.int64)
    for e, norm in enumerate(np.abs(const).sum(axis=-2).max(
            axis=-1, initial=0.0).astype(_f64)):
        bound, t = 1.0, 0
        while bound > 1e-24 or t <= orders + 2:
            t += 1
            bound *= norm / max(t - orders, 1)
        count[e] = t
    zero = np.zeros_like(const)
    term = [zero + np.eye(n, dtype=np.longdouble)] + [zero] * orders
    total = [zero.copy() for _ in range(orders + 1)]
    for t in range(1, count.max() + 1):
        new = []
        for k in range(orders + 1):
            v = times(cc, cv, term[k])
            if k:
                v += times(dc, dv, term[k - 1])
            new.append(v / t)
        term = new
        on = slice(None) if count.min() >= t else count >= t
        for k in range(orders + 1):
            total[k][on] += term[k][on]
    return total if extended else [m.astype(_f64) for m in total]


def coefficient_matrices(terms, drive, orders, extended=False):
    """E_0 .. E_orders of exp(sum_k scale_k M_k + f * drive) in powers of f
    for ``terms`` [(M_k, scale_k)].

    E_0 has the identity taken off.  Summed in extended precision and
    rounded once (not at all with ``extended``): the same E_k act at every
    step, so their rounding would not average out.
    """
    return [m[0] for m in coefficient_stacks([terms], drive, orders,
                                             extended)]


def chebyshev(mats, F):
    """Chebyshev coefficients in f / F of sum_k f^k E_k (not finite where a
    power of F is not)."""
    out = [np.zeros_like(mats[0]) for _ in mats]
    with np.errstate(over="ignore", invalid="ignore"):
        for k, m in enumerate(mats):
            power = np.zeros(k + 1)
            power[k] = _f64(F) ** k
            for j, c in enumerate(np.polynomial.chebyshev.poly2cheb(power)):
                if c:
                    out[j] += c * m
    return out


def scaled_powers(j, F):
    """(k, coefficient of f^k) of the Chebyshev polynomial T_j(f / F).

    Powers of F so small that the coefficient overflows are left out: the
    order-j part of a series at that F, which it would multiply, has
    underflowed to zero."""
    unit = np.zeros(j + 1)
    unit[j] = 1.0
    for k, c in enumerate(np.polynomial.chebyshev.cheb2poly(unit)):
        if c and F ** k and math.isfinite(float(c) / F ** k):
            yield k, c / F ** k


def economised(mats, da, db, F):
    """E_k with the Chebyshev polynomials of the orders that (da, db) leave
    out taken off, so that the kept ones represent the truncated Chebyshev
    series."""
    kept = [m.copy() for m in mats]
    cheb = chebyshev(mats, F)
    for j in _dropped(len(mats), da, db):
        for k, c in scaled_powers(j, F):
            kept[k] -= c * cheb[j]
    return kept


class SeriesModel:
    """E_k and row layout of one (constant, drive) pair at one step size.

    ``build`` returns None where the kernels do not apply: more than 64
    states, states the drive couples within a sector, sectors of more than
    ``SIZES`` components, a step whose constant part is large.
    """

    def __init__(self):
        self._tables = None     # the last drive's

    @classmethod
    def build(cls, const, drive, weights, h):
        """Model of the exponents h (w_j const + sum_s w_js c_s drive); one
        set of matrices per distinct w_j."""
        J, S = weights.shape
        sums = weights.sum(axis=1)
        if J not in (1, 2, 5) or (J <= 2 and S != J) or \
                not np.allclose(sums, sums[::-1], rtol=1e-15, atol=1e-16):
            return None
        self = cls.of_sets([[(const, h * float(w))]
                            for w in sums[:(J + 1) // 2]], drive, weights, h)
        if self is not None and J == 5 and self.size != SIZES[0]:
            return None
        return self

    @classmethod
    def of_sets(cls, sets, drive, weights, h, also=(), pair=False):
        """Model with one set of matrices per element of ``sets`` (terms of
        ``coefficient_matrices``) on sectors common to them and to ``also``
        (terms whose matrices are not needed).  ``pair``: None where
        ``one_pair`` does not hold."""
        n = drive.shape[0]
        if n > _lib.MAX_N:
            return None
        pattern = np.zeros((n, n))
        for terms in list(sets) + list(also):
            norm = sum(abs(s) * np.abs(m).sum(axis=0).max()
                       for m, s in terms)
            if not norm <= MAX_NORM:
                return None
            for m, _ in terms:
                pattern[m != 0] = 1.0
        found = split_sectors(pattern, drive)
        if found is None:
            return None
        sector, opposite = found
        counts = np.bincount(sector)
        fit = [s for s in SIZES if s >= counts.max()]
        if not fit:
            return None
        self = cls()
        self.n, self.size, self.h = n, fit[0], h
        self.sector, self.opposite = sector, opposite
        self.pad = fit[0] + 1                    # even
        self.n_sectors = counts.size
        self.weight = float(np.abs(weights).sum(axis=1).max())
        self.nnz = int(np.count_nonzero((pattern != 0) | (drive != 0)))
        order = np.argsort(sector, kind="stable")
        self.members = [order[np.searchsorted(sector[order], k):
                              np.searchsorted(sector[order], k, "right")]
                        for k in range(self.n_sectors)]
        pos = np.empty(n, dtype=np.int32)
        for k, states in enumerate(self.members):
            pos[states] = k * self.pad + np.arange(states.size)
        self.pos, self.order = pos, order
        if pair and not self.one_pair():
            return None
        top = 2 * ORDERS[-1][0] + 3
        self.stacks = coefficient_stacks(sets, drive, top)
        self.sets = [[m[e] for m in self.stacks] for e in range(len(sets))]
        return self

    def one_pair(self):
        """Whether one sector pair holds every state, so that a wavefront's
        lane rows can exchange without LDS."""
        return self.n_sectors <= 2 and \
            max(s.size for s in self.members) <= 11

    def flops(self, plan):
        """FP64 operations of one exponential: a multiply-add per order and
        entry of the sectors, two per row."""
        own = np.array([s.size for s in self.members])
        opp = np.where(self.opposite >= 0, own[self.opposite], 0)
        return int(2 * (own * (own * (plan[0] + 1) + opp * (plan[1] + 1) +
                               2)).sum())

    def plan(self, drive_max, tol, slope=None):
        """(da, db, F) for drives |c(t)| <= ``drive_max``, or None.

        F bounds the factors |f| and the kept orders are those of the
        series in Chebyshev polynomials of f / F, whose order k is 2^(k-1)
        smaller than the power series': what is left out must stay below
        ``tol`` with the Taylor plans' margin (a factor of 8).  With
        ``slope`` the derivative in f is used as well: of what is left out,
        it must stay below that share of the lowest even and odd order's.
        """
        F = self.h * self.weight * float(drive_max)
        worst = np.array([np.abs(c).sum(axis=-2).max()
                          for c in chebyshev(self.stacks, F)])
        if not np.all(np.isfinite(worst)):
            return None
        for da, db in ORDERS:
            left = _dropped(worst.size, da, db)
            # (the orders beyond the last matrix are smaller than it)
            if 8.0 * (worst[-1] + sum(worst[left])) > tol:
                continue
            # T_k' is k^2 at most, that of T_2 4, of T_1 1
            if slope is None or all(
                    sum(k * k * worst[k] for k in left if k % 2 == odd) <=
                    slope * lead
                    for odd, lead in ((0, 4 * worst[2]), (1, worst[1]))):
                return da, db, F
        return None

    def matrices(self, da, db, F):
        """The kept E_k of every set (``economised``)."""
        kept = economised(self.stacks, da, db, F)
        return [[m[e] for m in kept] for e in range(len(self.sets))]

    def tables(self, da, db, F):
        """(layout, on the host; device table) of the kernel's rows."""
        key = (da, db, F)
        # (another thread may keep its own drive's in between)
        kept = self._tables
        if kept is None or kept[0] != key:
            n, size = self.n, self.size
            layout = np.zeros((n, 4), dtype=np.int32)
            own_w, opp_w = size * (da + 1), size * (db + 1)
            sets = self.matrices(da, db, F)
            table = np.zeros((len(sets), own_w + opp_w, n))
            for r, state in enumerate(self.order):
                k = self.sector[state]
                o = self.opposite[k]
                layout[r] = (self.pos[state], k * self.pad,
                             (o if o >= 0 else k) * self.pad, state)
                for e, mats in enumerate(sets):
                    own = self.members[k]
                    for a in range(da + 1):
                        table[e, a:own.size * (da + 1):da + 1, r] = \
                            mats[2 * a][state, own]
                    if o < 0:
                        continue
                    opp = self.members[o]
                    for a in range(db + 1):
                        table[e, own_w + a:own_w + opp.size * (db + 1):
                              db + 1, r] = mats[2 * a + 1][state, opp]
            self._tables = kept = (key, layout, device_tensor(table))
        return kept[1:]

    def lane_tables(self, da, db, F, states):
        """Device (state per lane, table) of one instance per wavefront;
        ``states`` are the caller's indices of the model's."""
        lanes, own, opp = lane_entries(self)
        mats, = self.matrices(da, db, F)
        return (device_tensor(np.where(
            lanes >= 0, states[np.maximum(lanes, 0)], -1).astype(np.int32)),
            device_tensor(lane_table(mats, own, opp, da, db)))

    def shape(self, plan, whole=False):
        """The model's fields of ``ssmx_series_desc``; ``whole``: for the
        kernels of one instance per wavefront."""
        size = 11 if whole else self.size
        return dict(
            na=size, da=plan[0], nb=size, db=plan[1],
            sector=12 if whole else self.pad, sectors=self.n_sectors,
            sector_rows=self.members[0].size if self.n_sectors <= 2 else 0)


def lane_entries(model, transposed=False):
    """(state per lane, own entries, opposite entries) of one instance on a
    whole wavefront (``ssmx_series_queue``).

    An entry (slot, lane, row, column) names the matrix element the lane
    multiplies in that slot: of the own-sector tables, and of the tables
    that couple to the opposite sector.  ``transposed``: those of
    ``ssmx_series_adjoint``, whose lanes own columns.
    """
    lanes = np.full(64, -1, dtype=np.int32)
    own, opp = [], []
    pair = [model.members[0], model.members[1]
            if model.n_sectors > 1 else np.zeros(0, dtype=np.int64)]
    for lane in range(64):
        half, row, i = lane // 32, (lane // 16) % 2, lane % 16
        mine, other = pair[row], pair[1 - row]
        if i < mine.size:
            lanes[lane] = mine[i]
        for s in range(6 if half == 0 else 5):
            k = s + 6 * half
            if i < mine.size and k < mine.size:
                own.append((s, lane, mine[k], mine[i]) if transposed else
                           (s, lane, mine[i], mine[k]))
            # (tables of sectors that the drive leaves apart hold zeros there,
            # but a parameter's derivative may couple them)
            if transposed and i < mine.size and k < other.size:
                opp.append((s, lane, other[k], mine[i]))
            if not transposed and i < other.size and k < mine.size:
                opp.append((s, lane, other[i], mine[k]))
    return lanes, np.array(own, dtype=np.int64).reshape(-1, 4), \
        np.array(opp, dtype=np.int64).reshape(-1, 4)


def lane_table(mats, own, opp, da, db):
    """One set's table over ``lane_entries``."""
    out = np.zeros((6 * (da + 1) + 6 * (db + 1), 64))
    for k in range(da + 1):
        out[own[:, 0] * (da + 1) + k, own[:, 1]] = \
            mats[2 * k][own[:, 2], own[:, 3]]
    for k in range(db + 1):
        out[6 * (da + 1) + opp[:, 0] * (db + 1) + k, opp[:, 1]] = \
            mats[2 * k + 1][opp[:, 2], opp[:, 3]]
    return out


class SeriesRun:
    """Staged inputs of one run through ``ssmx_propagate_series``.

    ``states`` are the caller's indices of the model's states; ``rho0``
    (instances, n) and ``obs`` stay in the caller's order.  ``wave_group``
    consecutive instances share one waveform.
    """

    def __init__(self, model, plan, states, members, weights, nodes, rho0,
                 d_waves, d_segs, gen, fine, n_out, t0, dt, obs, read,
                 wave_group=1):
        torch = _torch()
        n_inst, n = rho0.shape
        flags = {"full": _lib.SSMX_READ_FULL, "obs": 0,
                 "integral": _lib.SSMX_READ_INTEGRAL}[read]
        n_obs = obs.shape[0] if obs is not None else 0
        if read != "full" and not 1 <= n_obs <= _lib.MAX_OBS:
            raise ValueError(f"{n_obs} readout rows outside 1.."
                             f"{_lib.MAX_OBS}")
        # a launch that leaves SIMDs idle spreads each instance over a whole
        # wavefront: 64 points of the 7-level sweep 344 -> 300 ns a step;
        # from two wavefronts per SIMD on, two instances to one are quicker
        # (ns a step: 1024 points 310 against 366, 1537 points 460 against 380)
        self.whole = members == 1 and model.one_pair() and \
            weights.shape[0] <= 2 and n_inst <= simd_count()
        states = np.asarray(states)
        if self.whole:
            self.layout, self.table = model.lane_tables(*plan, states)
        else:
            layout, self.table = model.tables(*plan)
            # the kernel's state index is the caller's
            layout = layout.copy()
            layout[:, 3] = states[model.order]
            self.layout = device_tensor(layout)
            where = np.full(n, -1, dtype=np.int32)
            where[states] = model.pos
            self.d_where = device_tensor(where)
        self.d_w, self.d_nodes = device_tensor(weights), device_tensor(nodes)
        self.d_rho0, self.d_waves, self.d_segs = (
            device_tensor(np.ascontiguousarray(rho0, dtype=_f64)), d_waves,
            d_segs)
        self.d_obs = None if read == "full" else device_tensor(
            np.ascontiguousarray(obs, dtype=_f64))
        self.desc = _lib.SeriesDesc(
            n=n, rows=model.n, n_inst=n_inst, members=members,
            n_exp=weights.shape[0], n_node=weights.shape[1], fine=fine,
            n_out=n_out, n_obs=n_obs, flags=flags, gen=gen,
            wave_group=wave_group, **model.shape(plan, self.whole),
            reserved=0, h=dt / fine, t0=t0, dt=dt)
        shape = {"full": (n_inst, n_out, n), "obs": (n_inst, n_out, n_obs),
                 "integral": (n_inst, n_obs)}[read]
        self.out = torch.empty(shape, dtype=torch.float64, device="cuda")
        self.k = members

    def launch(self):
        torch = _torch()
        stream = torch.cuda.current_stream().cuda_stream
        if self.whole:
            if self.desc.flags & _lib.SSMX_READ_FULL and \
                    self.desc.rows < self.desc.n:
                self.out.zero_()
            _lib.check(_lib.load().ssmx_propagate_series_wave(
                ctypes.byref(self.desc), _ptr(self.layout),
                _ptr(self.table), _ptr(self.d_w), _ptr(self.d_nodes),
                _ptr(self.d_waves), _ptr(self.d_segs), _ptr(self.d_rho0),
                _ptr(self.d_obs), _ptr(self.out), None,
                ctypes.c_void_p(stream)))
            return self.out
        _lib.check(_lib.load().ssmx_propagate_series(
            ctypes.byref(self.desc), _ptr(self.layout), _ptr(self.d_where),
            _ptr(self.table), _ptr(self.d_w), _ptr(self.d_nodes),
            _ptr(self.d_waves), _ptr(self.d_segs), _ptr(self.d_rho0),
            _ptr(self.d_obs), _ptr(self.out), ctypes.c_void_p(stream)))
        record_use(self.table)          # shared by the model's runs
        return self.out

    def result(self):
        return self.out
