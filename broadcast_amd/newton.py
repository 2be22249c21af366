"""Newton baseflow driver on the device (BROADCAST_npz.py:985-1196).

Per iteration, as the reference's `fixed_point` mode:

* boundary conditions, residual and its norms (compute_norml2inf);
* relaxation r = max over the first three variables of the norm ratios to
  the first iteration (:1062), coefdiag = r / dt * vol with
  dt = cfl (yc(1,2) - yc(1,1)) / (1/M + 1) (:1011-1012, :1063-1066), on the
  O-mesh dt = cfl |xc(1,2) - xc(1,1)| / (1/M + 1) (cylinder.py:842-894);
* the colored Jacobian -dR/dw + coefdiag, pruned, in CSR (:1068-1150);
* the linear solve J dw = R (MUMPS LU in the reference, :1152-1157; here the
  device block-banded LU below);
* w += dw.

Departures, each on the side of robustness: the reference runs a fixed
number of iterations, `newton` also stops when the residual norm
max_e ||R_e||_2 (compute_norml2, srcfv/norm.F90:2-32) falls below `tol`; on
a NaN step the reference subtracts the previous step and halves a cfl it no
longer uses (:1167-1172), `newton` restores the state before the step and
divides the cfl used for dt by `cfl_cut`, also when the residual norm grows
by more than `growth`.

Block-banded LU.  In the reference's unknown order (C-order ravel of
(im, jm, 5), i outermost) the Jacobian couples i-lines at most 3 apart, so it
is block banded with blocks of one i-line (5 jm unknowns).  The factorization
is block Gaussian elimination without pivoting across blocks, on the device by
the library's own kernels from both ends of the band (bca_band_factor): each
diagonal block is replaced by its inverse, the block rows by their products
with it; no fill leaves the band.  Storage is dense per block row,
R[K] = [A(K, K-kb) ... A(K, K+kb)], (nblocks, B, (2 kb + 1) B) doubles.
An i-periodic mesh (the O-mesh) couples the first and last i-lines; it is
solved with j outermost instead (blocks of one j-line), where the band is
that of the radial stencil.  Complex matrices, small pivots and CPU tensors
take torch's pivoted LU of the diagonal blocks.  The residual of a solve
(SOLVE_TOL) shows entries that grew in the elimination: solve(), or refine()
after it, then factors again, downwards only, then with the pivoted LU.
"""
from __future__ import annotations

import math
import time
from dataclasses import dataclass, field

import numpy as np

from . import device as dev

# A solve is corrected to a residual of REFINE_TOL times the right-hand side, at
# most REFINE_STEPS times.  Above SOLVE_TOL after that entries grew in the
# elimination, which chooses no pivot across the blocks (the pivots of its tiles
# do not show it), and the matrix is factored again a safer way: the Newton
# matrices end at 1e-12 to 1e-15, and 1e-8 still gives Newton its full step.
REFINE_TOL, REFINE_STEPS = 1e-12, 3
SOLVE_TOL = 1e-8


class BlockBandLU:
    """Dense block-banded LU on the device of an n x n CSR matrix whose
    unknown u = e + 5 (j + jm i) (0-based) is permuted to outer-major blocks.

    The band half-width kb (in blocks) is the widest coupling of every block
    row but the first: on the O-mesh (j-line blocks) the wall row j = 1 also
    reaches j = 5 (the off-centred Euler flux of the face j = 2), one block
    beyond the radial stencil's 3.  Such a far block of block row 0 is kept
    outside the band (eliminating block 0 turns it into in-band updates of
    block rows 1..kb), so the band stays 2 kb + 1 blocks wide: with kb = 3
    instead of 4, 9 instead of 16 Schur products per block step.

    With look-ahead (device tensors), the next diagonal block goes first and
    the remaining products of a step run beside it on another stream; the
    library's elimination then also works from both ends of the band at once."""

    def __init__(self, im, jm, outer="i", kb=None, group=1, lookahead=True, pivot=None, diag="inv", check=True):
        self.t = dev.torch()
        # pivot=None: the project's elimination without pivoting on the device
        # for the diagonal blocks -- diag="inv": their inverses by Gauss-Jordan
        # (bca_inv_np), the block row and the solves multiplied by them;
        # diag="lu": their LU factors (bca_lu_np) and triangular solves.
        # torch's pivoted LU on the CPU or when asked (pivot=True) or when a
        # pivot comes out too small.
        self.pivot = pivot
        if diag not in ("inv", "lu"):
            raise ValueError("diag must be 'inv' or 'lu'")
        self.diag = diag
        self.im, self.jm = im, jm
        self.outer = outer
        self.n = 5 * im * jm
        lines = im if outer == "i" else jm
        line = 5 * jm if outer == "i" else 5 * im
        self.B = group * line                      # unknowns per block: `group` outer lines
        self.nb = -(-lines // group)
        self.np = self.nb * self.B                 # padded with identity rows past n
        self.kb = kb
        self.lookahead = lookahead
        # check: solve() looks at its residual (a caller that gives every
        # solution to refine() leaves that to it)
        self.check = check
        self.ends = 2                              # ends of the band the elimination may work from
        self.mid = self.nb                         # block rows eliminated downwards (nb: all)

    def _perm(self, u):
        """Block-major index of the reference's unknown u."""
        if self.outer == "i":
            return u
        e = u % 5
        j = (u // 5) % self.jm
        i = u // (5 * self.jm)
        return e + 5 * (i + self.im * j)

    def factor(self, indptr, indices, data, shift=None):
        """Factor the CSR matrix (minus shift * I when shift is given): indptr
        of any integer type, its first entry that of indices and data."""
        t = self.t
        dv = data.device
        n, B = self.n, self.B
        self.csr = None
        counts = (indptr[1:] - indptr[:-1]).long()
        rows = self._perm(t.repeat_interleave(t.arange(n, device=dv), counts))
        cols = self._perm(indices.long())
        K, J = rows // B, cols // B
        d = J - K
        if self.kb is None:
            rest = K > 0
            kb = int(d[rest].abs().max()) if bool(rest.any()) else 0
            kb = max(kb, int((-d).max()), 1 if self.nb > 1 else 0)
            self.kb = min(kb, self.nb - 1)
        kb = self.kb
        far = d > kb
        if bool((far & (K > 0)).any()) or bool((d < -kb).any()):
            raise ValueError("entry outside the block band")
        self.nfar = int(d[far].max()) - kb if bool(far.any()) else 0
        if self.nfar > 1:
            # a far block two beyond the band would leave fill in block row 1
            # that the band does not hold
            self.kb = kb = kb + self.nfar - 1
            self.nfar, far = 1, d > kb
        W = (2 * kb + 1) * B
        inb = ~far
        R = t.zeros((self.nb, B, W), dtype=data.dtype, device=dv)
        R.view(-1).index_put_((((K * B + rows % B) * W + (d + kb) * B + cols % B)[inb],), data[inb])
        # far blocks of block row 0: columns kb+1 .. kb+nfar
        F = t.zeros((B, self.nfar * B), dtype=data.dtype, device=dv)
        if self.nfar:
            F.view(-1).index_put_((((rows % B) * (self.nfar * B) + (d - kb - 1) * B + cols % B)[far],), data[far])
        if shift is not None:
            u = t.arange(n, device=dv)
            R.view(-1)[((u // B) * B + u % B) * W + kb * B + u % B] -= shift
        if self.np > n:
            pad = t.arange(n, self.np, device=dv)
            R.view(-1)[((pad // B) * B + pad % B) * W + kb * B + pad % B] = 1.0
        self.R, self.F = R, F
        self.lu, self.piv = [None] * self.nb, [None] * self.nb
        # block Gaussian elimination: D_I = A(I, I) after the updates of the
        # steps before; X(I, J) = D_I^-1 A(I, J) stored in place of A(I, J);
        # A(K, J) -= A(K, I) X(I, J) for K, J in I+1..I+kb
        self.np_lu = self.pivot is not True and dv.type == "cuda" and data.dtype == t.float64
        if self.np_lu:
            self._bad = t.zeros(1, dtype=t.int32, device=dv)
            # solve() corrects with the matrix: a copy, the caller's arrays may
            # hold another one by then; queued before np_factor waits for its
            # result, so that a solve on any stream finds it complete
            if self.diag == "inv":
                self.csr, self.shift = csr_int32(indptr - indptr[:1], indices, data, copy=True), shift
            if self.np_factor(R, F):
                return self
            # a pivot came out too small
            self._safer()
            return self.factor(indptr, indices, data, shift)
        side = t.cuda.Stream() if (self.lookahead and dv.type == "cuda") else None
        cur = t.cuda.current_stream() if side is not None else None
        ready = None
        for I in range(self.nb):
            if ready is not None:
                cur.wait_event(ready)
                ready = None
            if self.lu[I] is None:
                self.lu[I], self.piv[I], _ = t.linalg.lu_factor_ex(R[I, :, kb * B:(kb + 1) * B])
            LU, piv = self.lu[I], self.piv[I]
            hi = min(I + kb, self.nb - 1)
            if hi == I:
                continue
            Xr = R[I, :, (kb + 1) * B:(kb + 1 + hi - I) * B]
            Xr.copy_(t.linalg.lu_solve(LU, piv, Xr))
            if I == 0 and self.nfar:
                F.copy_(t.linalg.lu_solve(LU, piv, F))
            # the next diagonal block first, then its factorization beside
            # the rest of this step's updates
            R[I + 1, :, kb * B:(kb + 1) * B].sub_(R[I + 1, :, (kb - 1) * B:kb * B] @ Xr[:, :B])
            if side is not None:
                ev = t.cuda.Event()
                ev.record(cur)
                side.wait_event(ev)
                with t.cuda.stream(side):
                    A1 = R[I + 1, :, kb * B:(kb + 1) * B]
                    self.lu[I + 1], self.piv[I + 1], _ = t.linalg.lu_factor_ex(A1)
                    ready = t.cuda.Event()
                    ready.record(side)
                self.lu[I + 1].record_stream(cur)
                self.piv[I + 1].record_stream(cur)
            for dd in range(1, hi - I + 1):
                K2 = I + dd
                L = R[K2, :, (kb - dd) * B:(kb - dd + 1) * B]
                if dd == 1:
                    # the diagonal block of K2 = I+1 is done: the blocks right of it
                    if hi - I > 1:
                        R[K2, :, (kb + 1) * B:(kb + hi - I) * B].sub_(L @ Xr[:, B:])
                else:
                    R[K2, :, (kb - dd + 1) * B:(kb - dd + 1 + hi - I) * B].sub_(L @ Xr)
                if I == 0 and self.nfar:
                    # far block f (absolute block kb + f) lies at offset kb + f - K2 of row K2
                    for f in range(1, self.nfar + 1):
                        off = kb + f - K2
                        if off <= kb:
                            R[K2, :, (kb + off) * B:(kb + off + 1) * B].sub_(L @ F[:, (f - 1) * B:f * B])
        if ready is not None:
            cur.wait_event(ready)
        return self

    def np_factor(self, R, F):
        """Block elimination with the project's unpivoted kernels: with
        diag="inv" the whole elimination is bca_band_factor (each diagonal
        block replaced by its inverse, from both ends of the band); with
        diag="lu" each diagonal block is replaced by its LU factors
        (bca_lu_np), the next one's on a side stream beside the rest of the
        step's products.  False if a pivot was too small."""
        self._bad.zero_()
        (self._factor_band if self.diag == "inv" else self._factor_lu)(R, F)
        return int(self._bad.item()) == 0

    def _factor_band(self, R, F):
        import ctypes as C
        from . import _lib

        t = self.t
        nb, B, kb = self.nb, self.B, self.kb
        # both ends need rows of their own beside the kb rows they meet in,
        # and the far blocks of block row 0 lie on its side
        # (they meet with the downward end kb steps behind: the upward end's
        # last kb steps come after it)
        self.mid = nb // 2 - kb
        if not self.lookahead or self.ends == 1 or self.mid < kb + self.nfar + 1:
            self.mid = nb
        scratch = t.empty(2 * (1 + kb + self.nfar) * B * B, dtype=t.float64, device=R.device)
        cur = t.cuda.current_stream()
        # the caller's stream may share a hardware queue with one of these:
        # it only waits for the two that do the work
        side = [t.cuda.Stream() for _ in range(2)] if self.lookahead else [cur] * 2
        streams = (C.c_void_p * 3)(*[s.cuda_stream for s in (cur, *side)])
        rc = _lib.lib().bca_band_factor(streams, C.c_void_p(R.data_ptr()), C.c_void_p(F.data_ptr()) if self.nfar else None,
                                        nb, B, kb, self.nfar, self.mid, C.c_void_p(scratch.data_ptr()), 1e-14,
                                        C.c_void_p(self._bad.data_ptr()))
        # the scratch and the matrix are in use on the other streams until the
        # caller's stream gets past them
        t.cuda.synchronize(R.device)
        _lib.check(rc, "bca_band_factor")

    def _factor_lu(self, R, F):
        import ctypes as C
        from . import _lib

        t = self.t
        B, kb = self.B, self.kb
        L_ = _lib.lib()
        W = R.shape[2]
        cur = t.cuda.current_stream()
        side = t.cuda.Stream() if self.lookahead else cur
        # scratch of each stream the diagonal blocks are processed on
        work = [t.empty(32 * 32, dtype=t.float64, device=R.device) for _ in range(2 if self.lookahead else 1)]

        def diag_np(I, stream):
            D = R[I, :, kb * B:(kb + 1) * B]
            wk = work[1 if (self.lookahead and stream is side) else 0]
            rc = L_.bca_lu_np(C.c_void_p(stream.cuda_stream), C.c_void_p(D.data_ptr()), B, W, 1e-14,
                              C.c_void_p(self._bad.data_ptr()), C.c_void_p(wk.data_ptr()))
            _lib.check(rc, "bca_lu_np")

        def apply_inv(D, X):
            """X <- D^-1 X in place."""
            X.copy_(t.linalg.solve_triangular(D, t.linalg.solve_triangular(D, X, upper=False, unitriangular=True),
                                              upper=True))

        diag_np(0, cur)
        ready = None
        for I in range(self.nb):
            if ready is not None:
                cur.wait_event(ready)
                ready = None
            hi = min(I + kb, self.nb - 1)
            if hi == I:
                continue
            D = R[I, :, kb * B:(kb + 1) * B]
            Xr = R[I, :, (kb + 1) * B:(kb + 1 + hi - I) * B]
            apply_inv(D, Xr[:, :B])
            R[I + 1, :, kb * B:(kb + 1) * B].sub_(R[I + 1, :, (kb - 1) * B:kb * B] @ Xr[:, :B])
            if self.lookahead:
                ev = t.cuda.Event()
                ev.record(cur)
                side.wait_event(ev)
                diag_np(I + 1, side)
                ready = t.cuda.Event()
                ready.record(side)
            else:
                diag_np(I + 1, cur)
            if hi - I > 1:
                apply_inv(D, Xr[:, B:])
            if I == 0 and self.nfar:
                apply_inv(D, F)
            for dd in range(1, hi - I + 1):
                K2 = I + dd
                L = R[K2, :, (kb - dd) * B:(kb - dd + 1) * B]
                if dd == 1:
                    if hi - I > 1:
                        R[K2, :, (kb + 1) * B:(kb + hi - I) * B].sub_(L @ Xr[:, B:])
                else:
                    R[K2, :, (kb - dd + 1) * B:(kb - dd + 1 + hi - I) * B].sub_(L @ Xr)
                if I == 0 and self.nfar:
                    for f in range(1, self.nfar + 1):
                        off = kb + f - K2
                        if off <= kb:
                            R[K2, :, (kb + off) * B:(kb + off + 1) * B].sub_(L @ F[:, (f - 1) * B:f * B])
        if ready is not None:
            cur.wait_event(ready)

    def _solve_diag(self, I, v):
        """D_I^-1 v for one block (v: (B,) or (B, k))."""
        t = self.t
        if not self.np_lu:
            return t.linalg.lu_solve(self.lu[I], self.piv[I], v.unsqueeze(1) if v.dim() == 1 else v).reshape(v.shape)
        kb, B = self.kb, self.B
        D = self.R[I, :, kb * B:(kb + 1) * B]
        m = v.unsqueeze(1) if v.dim() == 1 else v
        y = t.linalg.solve_triangular(D, t.linalg.solve_triangular(D, m, upper=False, unitriangular=True), upper=True)
        return y.reshape(v.shape)

    def solve(self, b):
        """x with A x = b, b in the reference's unknown order."""
        b = b.reshape(-1).contiguous()
        if self.np_lu and self.diag == "inv":
            check_vector(b, self.R)
            if not self.check or differentiated(b) or self.t.cuda.is_current_stream_capturing():
                return self._corrected(b)  # (a captured solve cannot ask for its residual)
            while self.np_lu:
                x, rel = self._settled(b)
                if rel <= SOLVE_TOL:
                    return x
                self.refactor()
        return self._apply(b)

    def _corrected(self, b):
        """The factors applied, and one correction with the matrix itself: the
        upward half of the elimination runs against the flow on a boundary
        layer, where (weakly relaxed) it loses some digits."""
        x = self._apply(b)
        return x + self._apply(self._residual(x, b))

    def _residual(self, x, b):
        r = csr_residual(self.csr, x, b)
        return r if self.shift is None else r + self.shift * x

    def _settled(self, b):
        """x and its residual relative to b, corrected as refine() does: while
        the residual is above REFINE_TOL and a correction halves it."""
        x = self._corrected(b)
        r, rel = self._rest(x, b)
        for _ in range(REFINE_STEPS):
            if rel <= REFINE_TOL:
                break
            y = x + self._apply(r)
            r, new = self._rest(y, b)
            if not new <= 0.5 * rel:
                break
            x, rel = y, new
        return x, rel

    def _rest(self, x, b):
        """b - A x, and its norm relative to b's (0 where that is none)."""
        r = self._residual(x, b)
        rn, bn = self.t.stack((r.norm(), b.norm())).tolist()
        return r, rn / bn if 0.0 < bn < math.inf else 0.0

    def _safer(self):
        """The next factorization's way: downwards only, as the flow runs, then
        with pivoting inside the diagonal blocks.  The present factors go."""
        if self.mid < self.nb:
            self.ends = 1
        else:
            self.pivot, self.kb = True, None
        self.R = self.F = None

    def refactor(self):
        """The same matrix factored again the next safer way; False where there
        is none."""
        if not self.np_lu or self.diag != "inv":
            return False
        self._safer()
        self.factor(*self.csr, shift=self.shift)
        return True

    def _apply(self, b):
        """The factors applied to b once."""
        t = self.t
        B, kb, nb = self.B, self.kb, self.nb
        if self.outer == "i":
            y = b.reshape(-1)
        else:
            y = b.reshape(self.im, self.jm, 5).permute(1, 0, 2).reshape(-1)
        y = t.cat((y, y.new_zeros(self.np - self.n))).reshape(nb, B)
        R = self.R
        if self.np_lu and self.diag == "inv":
            y = self._solve_band_torch(y) if differentiated(y) else self._solve_band(y)
            return self._unpermute(y)
        for I in range(nb):
            y[I] = self._solve_diag(I, y[I])
            for dd in range(1, min(kb, nb - 1 - I) + 1):
                y[I + dd] -= R[I + dd, :, (kb - dd) * B:(kb - dd + 1) * B] @ y[I]
        for I in range(nb - 1, -1, -1):
            for dd in range(1, min(kb, nb - 1 - I) + 1):
                y[I] -= R[I, :, (kb + dd) * B:(kb + dd + 1) * B] @ y[I + dd]
            if I == 0 and self.nfar:
                for f in range(1, self.nfar + 1):
                    if kb + f < nb:
                        y[0] -= self.F[:, (f - 1) * B:f * B] @ y[kb + f]
        return self._unpermute(y)

    def _solve_band(self, y):
        """bca_band_solve; y is overwritten."""
        import ctypes as C
        from . import _lib

        z = self.t.empty_like(y)
        _lib.check(_lib.lib().bca_band_solve(
            dev.current_stream_ptr(), C.c_void_p(self.R.data_ptr()),
            C.c_void_p(self.F.data_ptr()) if self.nfar else None, self.nb, self.B, self.kb, self.nfar, self.mid,
            C.c_void_p(y.data_ptr()), C.c_void_p(z.data_ptr())), "bca_band_solve")
        return z

    def _solve_band_torch(self, y):
        """bca_band_solve's products by torch, for derivatives through the solve."""
        nb, B, kb, mid, R = self.nb, self.B, self.kb, self.mid, self.R
        steps = [(I, range(I + 1, min(I + kb, nb - 1) + 1)) for I in range(mid)]
        if mid < nb:
            steps += [(I, range(I - kb, I)) for I in range(nb - 1, mid + kb - 1, -1)]
            steps += [(I, range(I + 1, mid + kb)) for I in range(mid, mid + kb)]

        def block(K, J):
            return R[K, :, (J - K + kb) * B:(J - K + kb + 1) * B]

        y, z = list(y.unbind(0)), [None] * nb
        for I, reach in steps:
            z[I] = block(I, I) @ y[I]
            for K in reach:
                y[K] = y[K] - block(K, I) @ z[I]
        for I, reach in reversed(steps):
            for K in reach:
                z[I] = z[I] - block(I, K) @ z[K]
            if I == 0:
                for f in range(1, min(self.nfar, nb - 1 - kb) + 1):
                    z[0] = z[0] - self.F[:, (f - 1) * B:f * B] @ z[kb + f]
        return self.t.stack(z)

    def _unpermute(self, y):
        y = y.reshape(-1)[:self.n]
        if self.outer == "i":
            return y
        return y.reshape(self.jm, self.im, 5).permute(1, 0, 2).reshape(-1)


def csr_int32(indptr, indices, data, copy=False):
    """The CSR as the kernels read it: int32 row starts and columns (torch's
    own CSR holds int64), each array consecutive."""
    t = dev.torch()
    indptr, indices = (a.to(t.int32, copy=copy).contiguous() for a in (indptr, indices))
    return indptr, indices, (data.clone() if copy else data).contiguous()


def check_vector(v, a):
    """The kernels read v as float64 values on the HIP device of the matrix a."""
    if v.dtype != dev.torch().float64 or v.device != a.device or not v.is_cuda:
        raise RuntimeError(f"expected float64 values on {a.device}, got {v.dtype} on {v.device}")


def differentiated(v):
    """Does torch take derivatives through v (or map over it)?  The kernels,
    which are given v's address, would leave it out."""
    t = dev.torch()
    if (v.requires_grad and t.is_grad_enabled()) or t.autograd.forward_ad.unpack_dual(v).tangent is not None:
        return True
    try:
        v.data_ptr()
    except RuntimeError:  # a transform's wrapper has no storage
        return True
    return False


def csr_residual(csr, x, b):
    """b - A x for the CSR (indptr, indices, data) on the device."""
    import ctypes as C
    from . import _lib

    t = dev.torch()
    indptr, indices, data = csr_int32(*csr)
    for a in (x, b, data):
        check_vector(a, indptr)
    if differentiated(x) or differentiated(b):
        counts = (indptr[1:] - indptr[:-1]).long()
        rows = t.repeat_interleave(t.arange(counts.numel(), device=data.device), counts)
        part = slice(int(indptr[0]), int(indptr[-1]))
        return b.index_add(0, rows, data[part] * x[indices[part].long()], alpha=-1)
    # the kernel reads both as consecutive values
    x, b = x.contiguous(), b.contiguous()
    r = t.empty_like(b)
    _lib.check(_lib.lib().bca_csr_residual(dev.current_stream_ptr(), b.numel(), C.c_void_p(indptr.data_ptr()),
                                           C.c_void_p(indices.data_ptr()), C.c_void_p(data.data_ptr()),
                                           C.c_void_p(x.data_ptr()), C.c_void_p(b.data_ptr()),
                                           C.c_void_p(r.data_ptr())), "bca_csr_residual")
    return r


def refine(lu, csr, b, x, rtol=REFINE_TOL, steps=REFINE_STEPS):
    """Iterative refinement of x (in place) for A x = b with the factors of
    lu, until ||b - A x|| <= rtol ||b||, a correction no longer halves the
    residual (its rounding floor), or `steps` corrections: the guard of the
    unpivoted factorization.  A residual left above SOLVE_TOL means that
    entries grew in it: lu factors again a safer way and x is solved anew.
    Returns (corrections, final relative residual)."""
    k, rel = correct(lu, csr, b, x, rtol, steps)
    while rel > SOLVE_TOL and lu.refactor():
        x.copy_(lu.solve(b))
        k, rel = correct(lu, csr, b, x, rtol, steps)
    return k, rel


def correct(lu, csr, b, x, rtol, steps):
    """refine()'s corrections with the factors as they are."""
    bn = float(b.norm())
    k = 0
    r = csr_residual(csr, x, b)
    rel = float(r.norm()) / max(bn, 1e-300)
    while rel > rtol and k < steps:
        dx = lu.solve(r)
        x += dx
        k += 1
        r = csr_residual(csr, x, b)
        new = float(r.norm()) / max(bn, 1e-300)
        if new > 0.5 * rel:
            rel = new
            break
        rel = new
    return k, rel


@dataclass
class NewtonLog:
    norms: list = field(default_factory=list)      # max_e ||R_e||_2 before each update
    relax: list = field(default_factory=list)      # r of each iteration
    seconds: list = field(default_factory=list)    # wall time of each iteration
    split: list = field(default_factory=list)      # per update: (jacobian, factor, solve) seconds
    refinements: list = field(default_factory=list)  # per update: (refinement steps, final relative residual)
    rollbacks: int = 0
    converged: bool = False


def interior(flow, a):
    """(im, jm, 5) view-copy of the interior of a flat state, the reference's
    unknown order after reshape(-1)."""
    return a.view(5, flow.nj, flow.ni)[:, 3:-3, 3:-3].permute(2, 1, 0).contiguous()


def newton(flow, w, ite=10, cfl=1e10, tol=1e-10, log=None, verbose=False, growth=1e3, cfl_cut=10.0, group=1):
    """The reference's Newton iteration on the flat device state w (updated
    in place).  Returns a NewtonLog."""
    t = dev.torch()
    log = NewtonLog() if log is None else log
    case = flow.case
    mach = case.phys.mach
    if case.kind == "cyl":
        # cylinder.py:842: |xc(1,2) - xc(1,1)|, the radial spacing at i = 1
        xc = flow.xc.view(flow.nj, flow.ni)
        dy = abs(float(xc[4, 3] - xc[3, 3]))
    else:
        # BROADCAST_npz.py:1011: yc(1,2) - yc(1,1), the first cell height
        yc = flow.yc.view(flow.nj, flow.ni)
        dy = float(yc[4, 3] - yc[3, 3])
    vol_int = flow.vol.view(flow.nj, flow.ni)[3:-3, 3:-3]      # (jm, im)
    res = flow.new_state()
    outer = "j" if case.kind == "cyl" else "i"
    norm0 = ninf0 = None
    w_prev, l2_prev = None, None
    it = 0
    while it < ite:
        it += 1
        t0 = time.perf_counter()
        flow.apply_bcs(w)
        res.zero_()
        flow.residual(w, res)
        norm, ninf = flow.norms(res)   # per variable sqrt(sum R^2) and (sum R^10)^(1/10)
        l2 = float(np.max(norm))
        if w_prev is not None and (not np.isfinite(l2) or l2 > growth * l2_prev):
            # rejected step: back to the previous state with a smaller cfl
            w.copy_(w_prev)
            cfl /= cfl_cut
            log.rollbacks += 1
            if verbose:
                print(f"newton it {it}: ||R|| = {l2:.3e} rejected, cfl -> {cfl:.3e}", flush=True)
            w_prev = None
            continue
        log.norms.append(l2)
        if verbose:
            print(f"newton it {it}: max ||R||_2 = {l2:.3e}", flush=True)
        if tol is not None and l2 < tol:
            log.converged = True
            log.seconds.append(time.perf_counter() - t0)
            break
        if norm0 is None:
            norm0 = 1.0 / np.maximum(norm, 1e-15)
            ninf0 = 1.0 / np.maximum(ninf, 1e-15)
        r = float(np.max([norm[:3] * norm0[:3], ninf[:3] * ninf0[:3]]))
        log.relax.append(r)
        dtm1 = (1.0 / mach + 1.0) / (cfl * dy)
        coefdiag = (r * dtm1 * vol_int).contiguous().reshape(-1)   # (im, jm) in Fortran order
        # the colored Jacobian straight into the pruned CSR; from the second
        # iteration on only the values are rewritten while every row keeps
        # its kept set (the same matrix as jacobian_colored + csr)
        indptr, indices, data = flow.jacobian_csr(w, coefdiag=coefdiag, refresh=True)
        t.cuda.synchronize()
        t1 = time.perf_counter()
        lu = BlockBandLU(flow.im, flow.jm, outer=outer, group=group, check=False).factor(indptr, indices, data)
        t.cuda.synchronize()
        t2 = time.perf_counter()
        rhs = interior(flow, res).reshape(-1)
        dw = lu.solve(rhs)
        log.refinements.append(refine(lu, (indptr, indices, data), rhs, dw))
        del lu
        w_prev, l2_prev = w.clone(), l2
        wi = w.view(5, flow.nj, flow.ni)[:, 3:-3, 3:-3]
        wi += dw.reshape(flow.im, flow.jm, 5).permute(2, 1, 0)
        t.cuda.synchronize()
        t3 = time.perf_counter()
        log.split.append((t1 - t0, t2 - t1, t3 - t2))
        log.seconds.append(t3 - t0)
    log.cfl = cfl
    return log


def continuation(flow_at, target, start, w=None, steps=4, ite=40, cfl=1e21, tol=1e-10, min_step=None, log=None,
                 verbose=False):
    """Continuation Newton in one flow parameter (the Reynolds number here):
    Newton at `start` (from w, or the free stream of flow_at(start)), then at
    parameters stepping to `target`, each solve starting from the previous
    baseflow; a step that does not converge is halved (down to min_step).
    flow_at(p) gives the Flow at parameter p on the same mesh.  Returns
    (flow at target, w at target, list of (p, NewtonLog)).  No reference
    counterpart: the reference's drivers start every solve from their own
    initial state."""
    from .flow import to_device

    t = dev.torch()
    f = flow_at(start)
    w = to_device(f.case.w) if w is None else w
    hist = []
    lg = newton(f, w, ite=ite, cfl=cfl, tol=tol)
    hist.append((start, lg))
    if not lg.converged:
        raise RuntimeError(f"continuation: no converged start at {start}")
    p = start
    dp = (target - start) / max(steps, 1)
    min_step = abs(dp) / 16 if min_step is None else min_step
    while (target - p) * np.sign(dp) > 1e-12:
        q = p + dp
        if (target - q) * np.sign(dp) < 1e-9 * abs(dp):
            q = target
        fq = flow_at(q)
        wq = w.clone()
        lq = newton(fq, wq, ite=ite, cfl=cfl, tol=tol)
        hist.append((q, lq))
        if verbose:
            print(f"continuation {p:.3g} -> {q:.3g}: {len(lq.norms) - 1} Newton steps, converged {lq.converged}",
                  flush=True)
        if lq.converged:
            p, w, f = q, wq, fq
        else:
            dp /= 2.0
            if abs(dp) < min_step:
                raise RuntimeError(f"continuation stalled at {p} (step {dp})")
        del wq
    t.cuda.synchronize()
    return f, w, hist
