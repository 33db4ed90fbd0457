"""Gradients through the series in the drive for models of 65 to 192 states.

The counterpart of ``SeriesGradient``: a forward run that stores every
exponential's input, a reverse run that stores the cotangents of the results,
and the contraction of their moments with d E_k / d theta
(``ssmx_series_wide_adjoint``, ``ssmx_series_moments``).
"""

import ctypes
import math

import numpy as np

from superspinsim_amd import _lib
from superspinsim_amd.propagator import _ptr, _torch, device_tensor
from superspinsim_amd.series import Reach
from superspinsim_amd.series_wide import WideModel, own_states

_f64 = np.float64

#: rows of the moment kernel
MAX_ROWS = 192
#: shares of the run's left-out entries that gradients try to leave out
FINER = (1e-1, 1.0)


def row_lists(mats):
    """(columns, values) [matrices][slots][n] of stacked matrices' rows."""
    m, n = mats.shape[0], mats.shape[1]
    width = int(np.max(np.count_nonzero(mats, axis=2), initial=0))
    at, row, col = np.nonzero(mats)
    # slot of each entry within its row
    key = at * n + row
    slot = np.arange(key.size) - np.searchsorted(key, key)
    cols = np.zeros((m, width, n), dtype=np.int32)
    vals = np.zeros((m, width, n))
    cols[at, slot, row] = col
    vals[at, slot, row] = mats[at, row, col]
    return cols, vals


class WideGradient:
    """Tables of one parameter point, or None from ``build`` where the
    kernels do not apply."""

    @classmethod
    def build(cls, sim, const, program, waves, dconst, rho0, obs, h, tol,
              adjoint_tol, derivatives):
        """Arguments as ``SeriesGradient.build``; ``derivatives`` unset: no
        backward will follow."""
        varying = [g for g in program if g is not None]
        if len(varying) != 1 or None not in program or sim.rotating or \
                sim.n <= _lib.MAX_N:
            return None
        folded, drive = sim.folded(const), sim.gens[varying[0]]
        pattern = (folded != 0) | (drive != 0)
        reach = Reach(pattern, rho0, np.atleast_2d(obs))
        states = reach.states
        if not _lib.MAX_N < states.size <= MAX_ROWS:
            return None
        at = np.ix_(states, states)
        c, g = folded[at], drive[at]
        model = WideModel.build(c, g, sim.weights, h)
        if model is None:
            return None
        plan = model.plan(max(w.abs_max()[varying[0]] for w in waves), tol)
        if plan is None:
            return None
        scale = h * float(sim.weights[0].sum())
        norm = scale * float(np.abs(c).sum(axis=0).max())
        # order k of a derivative is at most F^k |G|^k / k! e^norm |dA|, the
        # whole at least about e^-norm |dA|; four orders are kept, or three
        # where the quarter of the fourth that Chebyshev polynomials leave is
        # below the tolerance (a quarter less of the moments' work)
        b = plan[2] * float(np.abs(g).sum(axis=0).max())
        if not b <= 1.0:
            return None
        spread = math.exp(b + 2.0 * norm)
        if b ** 3 / 24.0 * spread <= adjoint_tol:
            orders = 3
        elif b ** 4 / 24.0 * spread <= adjoint_tol:
            orders = 4
        else:
            return None
        self = cls()
        self.model, self.plan, self.states = model, plan, states
        self.reach = reach
        self.orders = orders
        self.gen = program.index(varying[0])
        self.npad = -(-model.n // 16) * 16
        self.d_w, self.d_nodes = (device_tensor(sim.weights),
                                  device_tensor(sim.nodes))
        dc = dconst[:, at[0], at[1]]
        self.n_theta = dc.shape[0]
        if derivatives:
            self._stage_both()
            if self.back is None:
                return None
        else:
            self.tables = self._staged(model.layout(plan), states)
        if self.n_theta:
            order = np.argsort(model.pos)
            rows = np.ix_(order, order)
            terms, size = 4, 1.0
            while size > 1e-18:
                terms += 1
                size *= norm / (terms - 4)
            self.dtable = self._derivatives(
                scale * c[rows], g[rows],
                scale * dc[:, rows[0], rows[1]], terms, plan[2])
        return self

    @staticmethod
    def _staged(layout, states):
        if layout is None:
            return None
        blocks, lane_states, columns, table, in_lds = layout
        return blocks, device_tensor(own_states(lane_states, states)), \
            columns, table, in_lds

    def _stage_both(self):
        """Tables of the matrices and of their transposes (``back``: None
        where these don't fit), with as much of them as the kernel's columns
        hold in steps of ten: a gradient may hang on entries that the run
        itself is free to leave out."""
        da, db, F, budget = self.plan
        for share in FINER:
            self.plan = da, db, F, share * budget
            self.tables = self._staged(self.model.layout(self.plan),
                                       self.states)
            self.back = None if self.tables is None else self._staged(
                self.model.transposed(self.plan), self.states)
            if self.back is not None:
                return

    def _derivatives(self, a, g, da, terms, drive_max):
        """d E_k in every direction, by row position."""
        torch = _torch()
        n = a.shape[0]
        lists = []
        for mats in (a[None], g[None], da):
            col, val = row_lists(mats)
            lists.append((col.shape[1], device_tensor(col),
                          device_tensor(val)))
        out = torch.empty((da.shape[0], self.orders, self.npad, self.npad),
                          dtype=torch.float64, device="cuda")
        args = [v for s, col, val in lists
                for v in (ctypes.c_int32(s), _ptr(col), _ptr(val))]
        _lib.check(_lib.load().ssmx_series_derivatives(
            n, da.shape[0], terms, self.orders, drive_max, *args, _ptr(out),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        # (a backward may run on another stream than the setup)
        torch.cuda.current_stream().synchronize()
        return out

    def store_shape(self, n_inst, steps, J):
        """Inputs and cotangents of every exponential."""
        return 2, n_inst, steps, J, self.npad

    def _desc(self, problem, n_inst, in_lds):
        J, S = self.d_w.shape
        return _lib.SeriesDesc(
            n=problem.rho0.shape[-1], rows=self.model.n, n_inst=n_inst,
            members=1, n_exp=J, n_node=S, fine=problem.F,
            n_out=problem.n_out, n_obs=problem.obs.shape[0],
            flags=_lib.SSMX_READ_INTEGRAL, gen=self.gen, wave_group=1,
            lds_columns=in_lds, da=self.plan[0], db=self.plan[1],
            h=problem.dt / problem.F, t0=problem.t0, dt=problem.dt)

    def forward(self, problem, state, rho0, store):
        """Integrated readouts (n_inst, n_obs); ``store`` keeps the inputs
        of every exponential (or None)."""
        torch = _torch()
        n_inst = rho0.shape[0]
        out = torch.empty((n_inst, problem.obs.shape[0]),
                          dtype=torch.float64, device="cuda")
        factors = None
        if store is not None:
            factors = state.get("factors")
            shape = tuple(store.shape[1:4])
            if factors is None or tuple(factors.shape) != shape:
                factors = torch.empty(shape, dtype=torch.float64,
                                      device="cuda")
            state["factors"] = factors
        d_rho, d_obs = device_tensor(rho0), device_tensor(problem.obs)
        blocks, states, columns, table, in_lds = self.tables
        _lib.check(_lib.load().ssmx_propagate_series_wide(
            ctypes.byref(self._desc(problem, n_inst, in_lds)), _ptr(blocks),
            blocks.shape[0], _ptr(states), _ptr(columns), _ptr(table),
            _ptr(self.d_w), _ptr(self.d_nodes), _ptr(state["d_waves"]),
            _ptr(state["d_segs"]), _ptr(d_rho), _ptr(d_obs), _ptr(out),
            _ptr(store), _ptr(factors),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        self._keep = (d_rho, d_obs)
        return out

    def backward(self, problem, state, seed, g_theta, g_seg, lam):
        torch = _torch()
        n_inst = seed.shape[0]
        store, factors = state["inputs"], state["factors"]
        exps = store.shape[2] * store.shape[3]
        d_obs = device_tensor(problem.obs)
        if lam is not None:
            lam.zero_()
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        lib = _lib.load()
        blocks, states, columns, table, in_lds = self.back
        _lib.check(lib.ssmx_series_wide_adjoint(
            ctypes.byref(self._desc(problem, n_inst, in_lds)), _ptr(blocks),
            blocks.shape[0], _ptr(states), _ptr(columns), _ptr(table),
            _ptr(factors), _ptr(d_obs), _ptr(seed), _ptr(store[1]),
            _ptr(lam), stream))
        work = None
        if g_theta is not None and self.n_theta:
            work = torch.empty(
                (n_inst, lib.ssmx_series_moment_groups(
                    self.model.n, self.orders), self.n_theta),
                dtype=torch.float64, device="cuda")
            _lib.check(lib.ssmx_series_moments(
                self.model.n, n_inst, exps, self.orders, self.n_theta,
                _ptr(store[0]), _ptr(store[1]), _ptr(factors),
                _ptr(self.dtable), _ptr(work), _ptr(g_theta), stream))
        self._keep_back = (d_obs, seed, work)


__all__ = ["WideGradient", "row_lists"]
