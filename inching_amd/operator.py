"""Device operator for the eigensolvers: u = op(v) with op one of

* A v                                   (``Burn/Krylov/T3.py:54-239``)
* p(A) v, p the Chebyshev filter        (``Burn/PolynomialFilters/T2.py:28-92``)
* either of the above + shift Q^T Q v   (Hotelling / EED, ``Burn/Orthogonalization/T3.py:62-164``)

Precision policy: the block values and the Chebyshev recurrence vectors are float32 with
float32 accumulation in ``precision='f32'`` (mixed) mode and float64 in ``'f64'`` mode;
``'mf64'`` uses no stored values at all: the float64 ANM product is recomputed from the
float64 coordinates and the neighbour pattern (4 B of index traffic per neighbour instead
of 36-72 B of block values). v and u (the Lanczos basis side) are always float64. One
filtered matvec of degree m is m launches of the fused SpMV + three-term-recurrence kernel.

``timer``: optional list; when set, every operator launch is bracketed by HIP events on
the current stream and the event pairs are appended (kernel-time accounting).

With the matrix-free float64 operator, a filtered application runs its recurrence in slot
order (``BlockHessian.slot_form``: tiles, or records of the cluster layout): the input is
packed once next to the coordinates, the degree products read and write records, and the
accumulated result is unpacked once (``records=False`` or ``INCHING_RECORDS=0`` keeps the
vectors in the matrix's order).
"""
import os

import numpy as np
import torch

from . import ops

RECORDS = os.environ.get("INCHING_RECORDS", "1") != "0"


class Operator:
    def __init__(self, A, precision="f64", pol=None, Q=None, shift=0.0, lanes=None, timer=None, tune=True,
                 records=None):
        if precision not in ("f32", "f64", "mf64"):
            raise ValueError("precision must be 'f32', 'f64' or 'mf64'")
        self.A = A
        self.precision = precision
        self.timer = timer
        if precision == "mf64":
            self.vals = None
        else:
            A.ensure(precision)
            self.vals = A.vals(precision)
        self.n = A.shape[0]
        self.pol = pol
        self.Q = Q
        self.shift = float(shift)
        use_rec = RECORDS if records is None else bool(records)
        # a launch code for the matrix's order (other than the cluster layout's) asks for that order
        # (a code of the cluster layout's lays it out here, not inside a caller's capture)
        rec_ok = (pol is not None and precision == "mf64" and use_rec
                  and (lanes is None or (int(lanes) // 1000 & 4 and A.clusters() is not None))
                  and A.slot_form() is not None)
        if lanes is not None:
            self.lanes = int(lanes)
        elif rec_ok:
            self.lanes = None     # plain products only: picked when the first one comes
        elif tune:
            from .autotune import best_config
            self.lanes = best_config(A, precision)
        else:
            self.lanes = 161 if precision == "mf64" else A.lanes
        self.blanes, self.c16 = self.lanes, None
        if precision != "mf64":
            from .autotune import bsr_launch
            self.blanes, self.c16 = bsr_launch(A, self.lanes)
        self.n_spmv = 0
        self.n_apply = 0
        dev = A.device
        vdt = torch.float32 if precision == "f32" else torch.float64
        self.vdt = vdt
        if pol is not None:
            self._vk = torch.empty(self.n, dtype=vdt, device=dev)
            self._vkm1 = torch.empty(self.n, dtype=vdt, device=dev)
            self._vkp1 = torch.empty(self.n, dtype=vdt, device=dev)
            self._acc = torch.empty(self.n, dtype=vdt, device=dev)
            self.mu = [float(x) for x in pol.AdjustedCoefficients[:pol.AdjustedDegree + 1]]
            self.degree = int(pol.AdjustedDegree)
        self.rec = None
        if rec_ok:
            self.rec = A.slot_form()
            self._recs = self.rec.buffers(3)
            self._acc_rec = torch.empty(3 * self.rec.slots, dtype=torch.float64, device=dev)
            self._mu = np.array(self.mu, dtype=np.float64)
        if Q is not None:
            if Q.dtype != torch.float64 or Q.shape[1] != self.n:
                raise ValueError("Q must be float64 [m, 3N]")
            self.Q = Q.contiguous()
            self._h = torch.empty(Q.shape[0], dtype=torch.float64, device=dev)
            self._ws = ops.Workspace(Q.shape[0], dev)

    def spmv(self, x, y, _timed=True, **epi):
        timed = self.timer is not None and _timed
        if timed:
            e0 = torch.cuda.Event(enable_timing=True)
            e1 = torch.cuda.Event(enable_timing=True)
            e0.record()
        if self.vals is None:
            code = self.lanes
            if code is None:
                # the cluster layout (0.3 ms at 1,201 atoms, 16 at 2.4M) is laid out by the first product that can use
                # it; a capture cannot lay out anything, and takes the rows where no product came before
                code = 161
                if self.A.images is None and self.A._at_hand("_clusters"):
                    code = self.lanes = 161 if self.A.clusters() is None else 6001
            self.A.matfree_spmv(x, y, config=code, **epi)
        else:
            ops.bsr_spmv(self.A.n_atoms, self.A.rowptr, self.A.col, self.vals, x, y, lanes=self.blanes,
                         col16=self.c16, **epi)
        if timed:
            e1.record()
            epi = "cheb" if (epi.get("acc") is not None or epi.get("z") is not None) else "plain"
            self.timer.append((self.precision, epi, e0, e1, 1))
        self.n_spmv += 1

    def _filtered_records(self, v64, u64, shift=False):
        """u = sum_k mu_k T_k((A - cc)/dd) v with the recurrence on records: v packed into
        slot order, three record buffers in turn (T_k, T_{k-1} read, T_{k+1} written),
        the accumulator in slot order unpacked into u at the end (``shift``: with the Hotelling
        term added in the same launch)."""
        pol, form, acc = self.pol, self.rec, self._acc_rec
        ops.rec_pack(form.atoms, v64, self._recs[0], acc, self.mu[0])
        if self.timer is not None:
            e0 = torch.cuda.Event(enable_timing=True)
            e1 = torch.cuda.Event(enable_timing=True)
            e0.record()
        form.chebyshev(self._recs, self._mu, float(pol.cc), float(pol.dd), self.A.plus_i, acc)
        if self.timer is not None:
            e1.record()
            self.timer.append(("mf64rec", "cheb", e0, e1, self.degree))
        if shift:
            ops.shift_apply(self.Q, v64, -self.shift, u64, self._ws, atoms=form.atoms, acc=acc)
        else:
            ops.rec_unpack(form.atoms, acc, u64)
        self.n_spmv += self.degree

    def _on_records(self, v64, u64):
        return (self.rec is not None and v64.dtype == torch.float64 and u64.dtype == torch.float64
                and v64.is_contiguous() and u64.is_contiguous())

    def filtered(self, v64, u64):
        """u = sum_k mu_k T_k((A - cc)/dd) v.

        With a float64 operator the recurrence starts from v itself (it is only read) and,
        when u does not share v's memory, accumulates straight into u; otherwise v is
        converted into a scratch vector and the accumulator is converted into u at the end."""
        if self._on_records(v64, u64):
            self._filtered_records(v64, u64)
            return
        pol = self.pol
        dd, cc = float(pol.dd), float(pol.cc)
        scratch = [self._vk, self._vkm1, self._vkp1]
        f64 = self.vdt == torch.float64
        if f64 and v64.dtype == torch.float64 and v64.is_contiguous():
            cur = v64
        else:
            cur = scratch[0]
            ops.convert(v64, cur)
        direct = (f64 and u64.dtype == torch.float64 and u64.is_contiguous()
                  and u64.data_ptr() != v64.data_ptr())
        acc = u64 if direct else self._acc
        free = [b for b in scratch if b is not cur]
        ops.axpby(self.mu[0], v64, 0.0, acc)
        # the degree operator launches run back to back: one event pair times all of them
        if self.timer is not None:
            e0 = torch.cuda.Event(enable_timing=True)
            e1 = torch.cuda.Event(enable_timing=True)
            e0.record()
        prev = None
        for k in range(1, self.degree + 1):
            out = free.pop(0)
            if k == 1:
                self.spmv(cur, out, _timed=False, s1=1.0 / dd, c0=cc, acc=acc, mu=self.mu[1])
            else:
                self.spmv(cur, out, _timed=False, s1=2.0 / dd, c0=cc, z=prev, c2=1.0, acc=acc, mu=self.mu[k])
            if prev is not None and prev is not v64:
                free.append(prev)            # T_{k-2} v is no longer needed (v itself is never written)
            prev, cur = cur, out
        if self.timer is not None:
            e1.record()
            self.timer.append((self.precision, "cheb", e0, e1, self.degree))
        if not direct:
            ops.convert(acc, u64)

    def apply(self, v64, u64):
        self.n_apply += 1
        # a few rows Q (the six rigid motions) of a short vector and a result of its own: the Hotelling term in two
        # launches
        few = (self.Q is not None and self.shift != 0.0 and self.Q.shape[0] <= ops.SHIFT_MAX_M
               and self.n <= ops.SHIFT_MAX_DOF and v64.dtype == torch.float64 and u64.dtype == torch.float64 and v64.is_contiguous()
               and u64.is_contiguous() and v64.data_ptr() != u64.data_ptr())
        if few and self.pol is not None and self._on_records(v64, u64):
            self._filtered_records(v64, u64, shift=True)
            return u64
        if self.pol is None:
            self.spmv(v64, u64)
        else:
            self.filtered(v64, u64)
        if few:
            ops.shift_apply(self.Q, v64, -self.shift, u64, self._ws)
        elif self.Q is not None and self.shift != 0.0:
            m = self.Q.shape[0]
            ops.multidot(self.Q, m, v64, self._h, self._ws)
            ops.gemv_update(self.Q, m, self._h, u64, scale=-self.shift)
        return u64

    def plain(self, v64, u64):
        """A v without filter and without the Hotelling term."""
        self.spmv(v64, u64)
        return u64
